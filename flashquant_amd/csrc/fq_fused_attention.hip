// Fused TQ4 FlashAttention (prefill) for gfx950, head_dim 64, 128 and 256: un-rotated query in,
// packed TQ4 keys and values in, original-space output out.  (The figures in this comment are
// those of head_dim 128.)
//
// Operator: fused_tq_attention_reference
// (src/flashquant/kernels/cpu_reference.py:154-227) as dispatched by
// src/flashquant/kernels/attention.py:85-107:
//   q_rot = (q @ R^T) rounded to the query dtype
//   K, V  = centroid[idx] * norm in rotated space
//   out   = (softmax(q_rot K^T * scale + causal mask) V) @ R, rounded once
// The causal mask hides key j > query i counted from the top-left corner and is
// dropped when there is a single query row (cpu_reference.py:97-151).
//
// Work split.  A workgroup of 8 wavefronts serves one (batch, KV head) pair and 8
// "units": a unit is a block of 32 query positions of one query head of the group,
// so with 4 query heads per KV head a workgroup covers 64 positions of all 4 heads
// and every dequantised K/V tile is used for 256 query rows.
//
// Per 64-token tile all 512 threads dequantise K and V into LDS as fp16 with the
// norm folded in (one LDS lookup per packed byte in a byte -> (fp16, fp16) table),
// double buffered, one barrier per tile; then each wavefront runs
//   S^T (64 tokens x 32 rows)  = K_tile . q_rot^T      16 x v_mfma_f32_32x32x16_f16
//   O^T (128 coords x 32 rows) += V_tile^T . P^T        16 x v_mfma_f32_32x32x16_f16
// Both products are transposed so that a lane owns one query row (column l % 32 of
// every accumulator): the running maximum, the denominator and the rescale of O are
// per-lane scalars, and P goes from the S accumulator straight into the B operand
// of the second product.  That works because the contraction index of an MFMA may
// be permuted freely as long as both operands agree: the accumulator registers
// r = 8u .. 8u+7 of lane half hf hold rows 16u + 8a + 4hf + c (e = 4a + c), so the
// V tile stores token 16u + 8a + 4b + c at position 16u + 8b + 4a + c and a lane's
// 8 consecutive positions are exactly its 8 tokens.  The K tile uses the same
// permutation on the coordinates, and the query operand is read to match.
//
// head_dim 256: tiles of 32 tokens (the accumulators of 32 rows, their query operand and the scores are 208 of a lane's
// 256 registers, and 7 to 37 are spilled around the ends), the second product in groups of two coordinate blocks, the rotation
// matrix in four rounds through LDS (it is 256 KB in two terms).  Per flop the tile loop costs what it costs at 128: 2.6 us for
// 256 rows x 32 tokens, bound like it by the chain K reads - scores - weights - V reads - output.  The general kernel
// (fq_attention_any_dim.hip), which served this dimension with 16 rows a wavefront, read twice the LDS bytes per row: 2 x 32 x
// 700 tokens bf16 260 -> 110 us, 16 x 65 tokens 92 -> 51 us, 2 x 16 x 8192 tokens 4.11 -> 1.92 ms; in pieces 16 heads x 3001
// tokens fp16 516 -> 203 us, one query over 3 x 3500 tokens 350 -> 57 us.
//
// The two head rotations run inside the kernel (prologue and epilogue) on the fp16 MFMA
// with operands split into two fp16 terms, staged through the tile buffers.
#include "fq_common.hpp"
#include "fq_device.hpp"
#include "fq_attention_any_dim.hpp"
#include "fq_attention_expanded.hpp"
#include "fq_attention_schedule.hpp"

namespace fq {

// Tile geometry for head_dim D (64, 128 or 256).
template <int D>
struct PrefillCfg {
    static constexpr int TS = D == 256 ? 5 : 6;           // log2 of the tokens of a tile
    static constexpr int TT = 1 << TS;
    static constexpr int KSTRIDE = 2 * D + 16;            // bytes per token row of the K tile (D fp16 + pad): 4 banks
    static constexpr int KBYTES = TT * KSTRIDE;           // 17408 at D = 128
    static constexpr int VBYTES = 2 * D * TT;             // V^T tile: D coordinate rows x TT tokens fp16
    static constexpr int BUF = KBYTES + VBYTES;           // 33792 at D = 128
    static constexpr int NKS = D / 16;                    // k-steps of the score product
    static constexpr int NOB = D / 32;                    // 32-coordinate blocks of the output
    static constexpr int PB = D / 2;                      // packed bytes per token and head
    // The rotation matrix as MFMA operands (two fp16 terms), shared by the wavefronts of a workgroup:
    // a block of 32 x 16 holds one 16-byte operand per lane and term.  They lie where the tiles are between the query
    // stage and the end of the tile loop (64 KB), at D = 256 a quarter at a time, there and where the lookup tables are by turns.
    static constexpr int SLOT = 8 * (32 * D + 64);        // floats: per unit 32 rows un-normalised, 32 maxima, 32 sums
    static constexpr int RROUNDS = D == 256 ? 4 : 1;
    static constexpr int RBLK = NOB / RROUNDS;            // blocks of 32 result coordinates in a round
    static constexpr int RTERM = NKS * RBLK * 64 * 16;    // bytes per term: 32768 at D = 128 and 256
};

struct PrefillParams {
    const uint16_t* q;          // (B, H_Q, N_Q, 128)
    const uint8_t* k_packed;    // (B, H_KV, N_KV, 64)
    const float* k_norms;       // (B, H_KV, N_KV)
    const uint8_t* v_packed;
    const float* v_norms;
    const float* centroids_k;
    const float* centroids_v;
    const float* rotation;      // (128, 128)
    uint16_t* out;              // (B, H_Q, N_Q, 128)
    int rot_col_major;
    int H_Q, H_KV, G, N_Q, N_KV;
    int64_t k_cap, v_cap;       // tokens between the slabs of consecutive (batch, KV head) pairs (>= N_KV)
    int causal;
    float scale_log2e;
    // paged mode (variable-length queries over the packed paged cache)
    const int32_t* cu_seqlens_q;   // (S + 1,) first query token of every sequence in q / out (tokens, H_Q, 128)
    const int32_t* seq_lens;       // (S,) keys of every sequence, the new tokens included
    const int32_t* block_table;    // (S, max_blocks)
    const uint8_t* cache;          // (num_blocks, block_size, H_KV * 136)
    int max_blocks, num_blocks, bs_log2;
    int round_slots;               // workgroups running at a time (one per CU)
    // order and split of the work (fq_attention_schedule.hpp); workgroups in split pieces leave their rows in `part`
    int num_seqs, max_w, split_w, max_pieces;
    bool dense;                 // beyond kOrderSeqs sequences: max_w places for each of them
    bool all_in_part;           // workgroups that are not split leave their rows in `part` too
    float* part;                   // slot of a workgroup's piece: PrefillCfg<D>::SLOT floats
    int* left;                     // paged: pieces in `part` of every workgroup that may be split, 0 if none
    bool out_wide;                 // `out` is 16-byte aligned (its rows are multiples of 128 bytes apart)
};

__device__ __forceinline__ uint32_t scale_pair(uint32_t pair, half2v n2) {
    const half2v h = __builtin_bit_cast(half2v, pair) * n2;
    return __builtin_bit_cast(uint32_t, h);
}

template <bool PAGED>
__device__ __forceinline__ SeqShape seq_shape(const PrefillParams& p, int s) {
    int NQ = p.N_Q, NKV = p.N_KV, qoff = 0;
    if (PAGED) {
        NQ = p.cu_seqlens_q[s + 1] - p.cu_seqlens_q[s];
        NKV = p.seq_lens[s];
        const int room = p.max_blocks << p.bs_log2;
        NKV = NKV < 0 ? 0 : (NKV > room ? room : NKV);
        qoff = NKV - NQ > 0 ? NKV - NQ : 0;
    }
    return make_seq_shape(NQ, NKV, qoff, p.G, p.max_w);
}

// The sequences s0 + lane as the lanes of a wavefront hold them; empty ones past the end.
__device__ __forceinline__ SeqShape lane_shape(const PrefillParams& p, int s0, int lane) {
    // (no branch around the loads: the caller has other requests to send before it needs them)
    const bool some = s0 + lane < p.num_seqs;
    SeqShape sh = seq_shape<true>(p, some ? s0 + lane : p.num_seqs - 1);
    sh.NQ = some ? sh.NQ : 0;
    sh.NKV = some ? sh.NKV : 0;
    sh.qoff = some ? sh.qoff : 0;
    return make_seq_shape(sh.NQ, sh.NKV, sh.qoff, p.G, some ? p.max_w : 0);
}

// The share of a CU of the whole batch (all KV heads), in tiles, and the rows of the sequences that may be split.  The sums
// may wrap on batches beyond any memory: the pieces are then merely poor ones, and still the same everywhere.  `first`: the
// first wavefront's worth of sequences.
__device__ __forceinline__ BatchWork batch_work(const PrefillParams& p, const SeqShape& first, int lane) {
    uint32_t tiles = 0, rows = 0;
    for (int s0 = 0; s0 < p.num_seqs; s0 += kWave) {
        const SeqShape sh = s0 == 0 ? first : lane_shape(p, s0, lane);
        if (sh.W > 0)
            tiles += uint32_t(sh.W) * uint32_t(tiles_of(sh, 0, p.G, p.causal) + tiles_of(sh, sh.W - 1, p.G, p.causal) + 1) / 2;
        if (sh.W <= p.split_w) rows += uint32_t(sh.NQ) * uint32_t(p.G);
    }
    return {share_of(wave_sum(tiles) * uint32_t(p.H_KV), p.round_slots), int(wave_sum(rows) * uint32_t(p.H_KV) >> 8)};
}

// Pieces of a sequence's workgroups.
template <int D>
__device__ __forceinline__ int pieces_in(const PrefillParams& p, const SeqShape& sh, const BatchWork& batch) {
    return pieces_of(sh, batch, p.split_w, p.max_pieces, p.G, p.causal != 0, D);
}

struct WorkItem {
    int seq, x, piece, pieces;      // seq < 0: none
};

// What the combine needs to know of its workgroup `at`, so that one without work costs a load (adding up the lengths there
// took 5 us a launch).  The grid has more workgroups than there are such entries.
template <int D>
__device__ __forceinline__ void note_pieces(const PrefillParams& p, const SeqShape& first, const BatchWork& batch, int at, int lane) {
    if (at >= p.num_seqs * p.H_KV * p.split_w) return;
    const int x = at % p.split_w, b = at / p.split_w / p.H_KV;
    auto of_lane = [&](int v) { return __builtin_amdgcn_readlane(v, b); };
    const SeqShape sh = b < kWave ? make_seq_shape(of_lane(first.NQ), of_lane(first.NKV), of_lane(first.qoff), p.G, p.max_w)
                                  : seq_shape<true>(p, b);
    const int n = x < sh.W && sh.W <= p.split_w ? pieces_in<D>(p, sh, batch) : 0;
    if (threadIdx.x == 0) p.left[at] = n > 1 || p.all_in_part ? n : 0;
}

// Contiguous sequences, all of one shape and in as many pieces as the host has worked out: the workgroups of all of them from
// the last one down.
__device__ __forceinline__ WorkItem find_prompt_item(const PrefillParams& p, int at) {
    const int place = at / p.H_KV, per = p.num_seqs * p.max_pieces, down = place / per, rest = place % per;
    const int W = seq_shape<false>(p, 0).W;
    if (down >= W) return WorkItem{-1, 0, 0, 1};
    return WorkItem{rest / p.max_pieces, W - 1 - down, rest % p.max_pieces, p.max_pieces};
}

// The item of a place (`at` / H_KV, of one KV head) of a paged batch in the order longest piece first: the largest tile count
// T that more than `place` pieces reach, a lane per sequence, three counts at a time (they do not wait for one another) between
// 0 and the longest context; then the place among the pieces of exactly T.  Beyond kOrderSeqs sequences the items in the order
// of the sequences (kOrderSeqs says why).  SPLIT: `at` is the workgroup's number in the launch.  `first`: the first wavefront's
// worth of sequences.
template <int D, bool SPLIT>
__device__ __forceinline__ WorkItem find_item(const PrefillParams& p, int at, const SeqShape& first, int lane) {
    const int G = p.G, place = at / p.H_KV;
    const bool causal = p.causal != 0;
    if (p.dense) {
        const int seq = place / p.max_w, x = p.max_w - 1 - place % p.max_w;
        return seq < p.num_seqs && x < seq_shape<true>(p, seq).W ? WorkItem{seq, x, 0, 1} : WorkItem{-1, 0, 0, 1};
    }
    // (the lengths of the batch are only summed where a sequence is long enough for the shortest pieces)
    BatchWork batch{kSplitMinTiles, 0};
    if (SPLIT && (p.num_seqs > kWave || __any(may_split(first, p.split_w, p.max_pieces, G, causal, D))))
        batch = batch_work(p, first, lane);
    if (SPLIT) note_pieces<D>(p, first, batch, at, lane);
    auto shape = [&](int s0) { return s0 == 0 ? first : lane_shape(p, s0, lane); };
    const int first_pieces = SPLIT ? pieces_in<D>(p, first, batch) : 1;
    auto pieces = [&](int s0, const SeqShape& sh) { return s0 == 0 || !SPLIT ? first_pieces : pieces_in<D>(p, sh, batch); };
    struct Counts { int c[3]; };
    auto count = [&](int t0, int t1, int t2) {           // pieces of at least so many tiles
        uint32_t c0 = 0, c1 = 0, c2 = 0;
        for (int s0 = 0; s0 < p.num_seqs; s0 += kWave) {
            const SeqShape sh = shape(s0);
            const int n = pieces(s0, sh);
            c0 += uint32_t(n * (sh.W - first_piece_with(sh, t0, n, G, causal)));
            c1 += uint32_t(n * (sh.W - first_piece_with(sh, t1, n, G, causal)));
            c2 += uint32_t(n * (sh.W - first_piece_with(sh, t2, n, G, causal)));
        }
        return Counts{{int(wave_sum(c0)), int(wave_sum(c1)), int(wave_sum(c2))}};
    };
    WorkItem item{-1, 0, 0, 1};
    int lo = 0, hi = 0x3fffffff, rem = place;            // tile counts lo .. hi - 1 (no sequence has 2^30 tiles)
    if (p.num_seqs <= kOrderSeqs) {
        float most = 0.0f;                               // (rounded up past 2^24)
        for (int s0 = 0; s0 < p.num_seqs; s0 += kWave) most = __builtin_fmaxf(most, float(shape(s0).all_tiles));
        hi = __builtin_amdgcn_readfirstlane(int(wave_max(most) * 1.000001f)) + 1;
        int at_hi = 0;                                   // count(lo) > place >= count(hi)
        if (place >= count(0, 0, 0).c[0]) return item;
        while (hi - lo > 1) {
            const int m1 = (lo + hi) >> 1, m0 = (lo + m1) >> 1, m2 = (m1 + hi) >> 1;
            const Counts c = count(m0, m1, m2);
            const int below = c.c[1] > place ? 2 : 0;    // which half, then which quarter
            const int mid = c.c[1] > place ? m2 : m0, at_mid = c.c[below];
            if (c.c[1] > place) lo = m1;
            else { hi = m1; at_hi = c.c[1]; }
            if (at_mid > place) lo = mid;
            else { hi = mid; at_hi = at_mid; }
        }
        rem = place - at_hi;
    }
    for (int s0 = 0; s0 < p.num_seqs; s0 += kWave) {
        const SeqShape sh = shape(s0);
        const int n = pieces(s0, sh), x0 = first_piece_with(sh, lo, n, G, causal);
        const int mine = n * (first_piece_with(sh, hi, n, G, causal) - x0);
        int before = mine;            // pieces of the lanes up to this one
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const int v = __shfl_up(before, d, kWave);
            if (lane >= d) before += v;
        }
        const uint64_t hit = __ballot(rem < before);
        if (hit != 0) {
            const int l = __ffsll(static_cast<unsigned long long>(hit)) - 1;
            const int at = rem - (__builtin_amdgcn_readlane(before, l) - __builtin_amdgcn_readlane(mine, l));
            item.pieces = __builtin_amdgcn_readlane(n, l);
            item.seq = s0 + l;
            item.piece = at % item.pieces;
            item.x = __builtin_amdgcn_readlane(x0, l) + at / item.pieces;
            return item;
        }
        rem -= __builtin_amdgcn_readlane(before, kWave - 1);
    }
    return item;
}

// The rotation matrix as the A operand of v_mfma_f32_32x32x16_f16, split once per workgroup.
// Both rotations are transposed products, matrix block x row block: a lane then owns one query row in
// the operand (its own 16-byte pieces of the query, or its registers of O) and in the result, and no row
// passes through LDS.  Block (32 result coordinates, 16 contraction coordinates): lane (m32, hf) holds
// eight contraction coordinates of result coordinate m32, as two fp16 terms.  Wavefront w fetches and
// splits blocks BPW * w .., every wavefront reads all of them.
//
// What it replaced staged the rows through LDS for the 16x16x32 MFMA (16 to 32 lanes on a bank) and stored the
// results 2 bytes a lane: a workgroup per CU on 64 tokens of 32 heads over 64 keys took 33 us and 27 us with one
// query row, 24 and 15.5 us this way (the tile itself: 2 us); 4 x 32 heads x 8192 tokens 2.89 -> 2.81 ms.
//
// At 256 coordinates the matrix comes in rounds.  AREAS: 2 where they take turns in two places, 1 where each waits for the one
// before to be done with (attention_combine_prompts_kernel).
template <int D, int AREAS = 2>
struct RotationBlocks {
    using Cfg = PrefillCfg<D>;
    static constexpr int NKS = Cfg::NKS, RBLK = Cfg::RBLK, BPW = RBLK * NKS / 8;
    static constexpr int RROUNDS = Cfg::RROUNDS;
    const float* rotation;
    bool col_major;
    uint8_t* share;               // 2 x RTERM bytes of LDS: the last round's operands, and every second one's before it
    uint8_t* other;               // as many again for the rounds between (unused with one round, or one area)
    int w, lane, m32, hf;
    float rbv[BPW][8];
    // `back`: x @ R with the contraction index in the order of the accumulator registers (element 4 a + c of half
    // hf = coordinate 8 a + 4 hf + c of the k-step), else x @ R^T in the natural order
    __device__ __forceinline__ void fetch(bool back, int round) {
#pragma unroll
        for (int i = 0; i < BPW; ++i) {
            const int blk = BPW * w + i, j = 32 * (RBLK * round + blk / NKS) + m32, k0 = 16 * (blk % NKS);
            const int k1 = back ? k0 + 4 * hf : k0 + 8 * hf, step = back ? 8 : 4;    // coordinates k1 + 0..3, k1 + step + 0..3
            if (back == col_major) {                       // a lane's coordinates are neighbours in memory
                const float4v lo = *reinterpret_cast<const float4v*>(rotation + j * D + k1);
                const float4v hi = *reinterpret_cast<const float4v*>(rotation + j * D + k1 + step);
#pragma unroll
                for (int e = 0; e < 4; ++e) { rbv[i][e] = lo[e]; rbv[i][4 + e] = hi[e]; }
            } else {                                       // the lanes' are
#pragma unroll
                for (int e = 0; e < 8; ++e) rbv[i][e] = rotation[(k1 + (e >> 2) * step + (e & 3)) * D + j];
            }
        }
    }
    __device__ __forceinline__ uint8_t* at(int round) const { return AREAS == 1 || ((RROUNDS - 1 - round) & 1) == 0 ? share : other; }
    __device__ __forceinline__ void put(int round) {
        uint8_t* dst = at(round);
        half8 rhi[BPW], rlo[BPW];
        split_rotation_block<32 * BPW>(rbv, rhi, rlo);
#pragma unroll
        for (int i = 0; i < BPW; ++i) {
            *reinterpret_cast<half8*>(dst + ((BPW * w + i) * 64 + lane) * 16) = rhi[i];
            *reinterpret_cast<half8*>(dst + Cfg::RTERM + ((BPW * w + i) * 64 + lane) * 16) = rlo[i];
        }
    }
    // The products of a round with this wavefront's 32 rows (`a`, and with ROWS_LO `alo`, 2^12 times what `a` leaves of
    // them); done(block of the round, high sums, low sums times 2^12).  The matrix operands are read two groups of two k-steps
    // (one at 256 coordinates, where registers are few) ahead of their products: the compiler on its own reads one product
    // ahead.  The fences hold LDS reads and products in this order and let the vector instructions of the block before pass.
    // Bound by LDS: eight wavefronts read the 64 KB of a round each, 3.4 us at the 150 bytes a ns that a CU's LDS gives here.
    template <bool ROWS_LO, class Done>
    __device__ __forceinline__ void products(int round, const half8 (&a)[NKS], const half8 (&alo)[NKS], const Done& done) const {
        constexpr int GK = D == 256 ? 1 : 2, GROUPS = NKS / GK, ALL = RBLK * GROUPS, kFence = 0x76;
        const uint8_t* src = at(round) + 16 * lane;
        half8 t[ALL][2][GK];
        auto read = [&](int g) {
#pragma unroll
            for (int k = 0; k < GK; ++k)
#pragma unroll
                for (int term = 0; term < 2; ++term)
                    t[g][term][k] = *reinterpret_cast<const half8*>(src + term * Cfg::RTERM + (GK * g + k) * 1024);
        };
        read(0);
        read(1);
        __builtin_amdgcn_sched_barrier(kFence);
        float16v hi, lo;
#pragma unroll
        for (int g = 0; g < ALL; ++g) {
            if (g + 2 < ALL) {
                read(g + 2);
                __builtin_amdgcn_sched_barrier(kFence);
            }
            if (g % GROUPS == 0)
#pragma unroll
                for (int r = 0; r < 16; ++r) { hi[r] = 0.0f; lo[r] = 0.0f; }
#pragma unroll
            for (int k = 0; k < GK; ++k) {
                const int ks = GK * (g % GROUPS) + k;
                hi = __builtin_amdgcn_mfma_f32_32x32x16_f16(t[g][0][k], a[ks], hi, 0, 0, 0);
                lo = __builtin_amdgcn_mfma_f32_32x32x16_f16(t[g][1][k], a[ks], lo, 0, 0, 0);
                if (ROWS_LO) lo = __builtin_amdgcn_mfma_f32_32x32x16_f16(t[g][0][k], alo[ks], lo, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(kFence);
            if (g % GROUPS == GROUPS - 1) done(g / GROUPS, hi, lo);
        }
    }
};

// The end of a workgroup: the rows in the accumulators normalised, rotated back (the first round of the matrix already lies
// in LDS) and stored.  EARLY: with two areas the second round is asked for before the rows are converted, else after.
template <int D, int DT, bool PAGED, bool EARLY, int AREAS>
__device__ __forceinline__ void finish_rows(const PrefillParams& p, RotationBlocks<D, AREAS>& rot, float16v (&O)[D / 32], float inv,
                                            bool unit_live, int pos0, int hq, int NQ, int64_t q_row0, int q_stride) {
    using Cfg = PrefillCfg<D>;
    constexpr int NKS = Cfg::NKS, NOB = Cfg::NOB, RROUNDS = Cfg::RROUNDS, RBLK = Cfg::RBLK;
    const int m32 = rot.m32, hf = rot.hf;
    if (RROUNDS == 1 && !unit_live) return;
    if (RROUNDS > 1 && AREAS > 1 && EARLY) rot.fetch(true, 1);
    // float32 rows: both operands as two fp16 terms, three MFMA terms; rows already rounded to 16 bits (the paged form) in
    // one, the row's largest value brought into [2^14, 2^15): what is above 2^-28 of it is exact, the rest to 2^-39 of it (a
    // largest value in [1, 2) left the coordinates below 2^-14 of it among fp16's subnormals)
    constexpr int kUp = PAGED ? 14 : 0;
    float mo = 0.0f;
#pragma unroll
    for (int ob = 0; ob < NOB; ++ob)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float v = O[ob][r] * inv;
            O[ob][r] = PAGED ? load_elem<DT>(store_elem<DT>(v)) : v;
            mo = __builtin_fmaxf(mo, __builtin_fabsf(O[ob][r]));
        }
    const int eo = row_exponent(mo);
    half8 ohi[NKS], olo[NKS];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const float a0 = O[ks >> 1][8 * (ks & 1) + e] * pow2(kUp - eo), a1 = O[ks >> 1][8 * (ks & 1) + e + 1] * pow2(kUp - eo);
            if (PAGED) {
                ohi[ks][e] = _Float16(a0); ohi[ks][e + 1] = _Float16(a1);
            } else {
                const auto h2 = __builtin_amdgcn_cvt_pkrtz(a0, a1);
                const auto l2 = __builtin_amdgcn_cvt_pkrtz((a0 - float(h2[0])) * 4096.0f, (a1 - float(h2[1])) * 4096.0f);
                ohi[ks][e] = h2[0]; ohi[ks][e + 1] = h2[1];
                olo[ks][e] = l2[0]; olo[ks][e + 1] = l2[1];
            }
        }
    if (RROUNDS > 1 && AREAS > 1 && !EARLY) rot.fetch(true, 1);
    const int opos = pos0 + m32;
    uint16_t* obase = PAGED ? p.out + (q_row0 + hq) * D : p.out + (q_row0 + int64_t(hq) * NQ) * D;
    uint16_t* orow = obase + int64_t(opos) * q_stride;
#pragma unroll
    for (int round = 0; round < RROUNDS; ++round) {
        if (round > 0) __syncthreads();                // the operands before are done with; with two areas this round's are there
        if constexpr (AREAS == 1) {
            if (round > 0) {
                rot.put(round);
                __syncthreads();
            }
            if (round + 1 < RROUNDS) rot.fetch(true, round + 1);
        } else {
            if (round + 1 < RROUNDS) rot.put(round + 1);
            if (round + 2 < RROUNDS) rot.fetch(true, round + 2);
        }
        rot.template products<!PAGED>(round, ohi, olo, [&](int cr, const float16v& hi, const float16v& lo) {
        const int cb = RBLK * round + cr;
        // registers 4 q + c of half hf = coordinate 32 cb + 8 q + 4 hf + c; the halves exchange a quad of every two,
        // so that a lane stores eight neighbours at a time
        uint32_t wd[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float v0 = (hi[2 * i] + lo[2 * i] * (1.0f / 4096.0f)) * pow2(eo - kUp);
            const float v1 = (hi[2 * i + 1] + lo[2 * i + 1] * (1.0f / 4096.0f)) * pow2(eo - kUp);
            wd[i] = uint32_t(store_elem<DT>(v0)) | uint32_t(store_elem<DT>(v1)) << 16;
        }
#pragma unroll
        for (int q = 0; q < 4; q += 2) {
            const auto x = __builtin_amdgcn_permlane32_swap(wd[2 * q], wd[2 * q + 2], false, false);
            const auto y = __builtin_amdgcn_permlane32_swap(wd[2 * q + 1], wd[2 * q + 3], false, false);
            const uint4v v = {x[0], y[0], x[1], y[1]};
            uint16_t* dst = orow + 32 * cb + 8 * q + 8 * hf;
            if (opos < NQ && unit_live) {
                if (p.out_wide) {
                    *reinterpret_cast<uint4v*>(dst) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        dst[2 * e] = uint16_t(v[e] & 0xffffu);
                        dst[2 * e + 1] = uint16_t(v[e] >> 16);
                    }
                }
            }
        }
        });
    }
}

// Where a workgroup's work comes from and what becomes of its rows.  At 256 coordinates the end of a workgroup beside the
// branch that leaves its rows to the combine costs 157 to 195 spilled registers, some of them inside the tile loop, either
// one alone 7 to 37: 8 sequences of 120 queries over 1500 keys, 32 heads, 226 us with both compiled in, 170 with one.
enum Work {
    kGrid,            // one workgroup per grid position, rows finished in the kernel
    kOrdered,         // find_item, the same (paged)
    kPieces,          // find_item, rows of a piece left to the combine, other rows finished in the kernel (paged)
    kAllPieces        // find_item or find_prompt_item, all rows left to the combine
};

// PAGED: the sequences' queries are packed along the token axis of q (tokens, H_Q, 128), the keys
// and values come from the paged TQ4 cache through the block table, query j of a sequence with
// n queries and L keys sits at position L - n + j (the new tokens are the last ones), and the
// attention result is rounded to the query dtype before the rotation back, as the attention
// library's output is in the path this replaces (src/flashquant/vllm/impl.py:265-336, 470-512).
// WORK: how the workgroups take their work and where it ends (below).
template <int D, int DT, bool PAGED, int WORK>
__global__ __launch_bounds__(512) void fused_tq_attention_kernel(const PrefillParams p) {
    using Cfg = PrefillCfg<D>;
    constexpr int kPfKStride = Cfg::KSTRIDE, kPfKBytes = Cfg::KBYTES, kPfBufBytes = Cfg::BUF;
    constexpr int NKS = Cfg::NKS, NOB = Cfg::NOB, PB = Cfg::PB, TS = Cfg::TS, TT = Cfg::TT;
    constexpr int NTB = TT / 32, NVS = TT / 16;    // 32-token blocks of the scores, k-steps of the second product
    constexpr bool kFind = WORK != kGrid, kSplit = WORK == kPieces || WORK == kAllPieces;
    // In grid order there is no search to hide the matrix behind, and at 64 coordinates the values held meanwhile and the way
    // round the products cost more than they give: bf16, causal, 32 heads over 8, 2 x 8192 tokens 949 us with them and 927
    // without, 4 x 1500 106.8 and 104.6, 16 x 300 42.9 and 42.0.  At 256 the second round of the matrix at the end is asked for
    // behind the conversions, not before them (2 x 8192 tokens, 16 heads over 4, 2.00 ms with 56 spilled registers and 1.92 with
    // 26, one prompt of them 1175 and 1154, 8 x 500 of 32 over 8 165 and 156); the other forms spill 7 to 37 either way and
    // gain by it (one prompt of 3001 in pieces 381 and 377).
    constexpr bool kEarlyFetch = kFind || D != 64, kSkipDead = kFind || D != 64, kEarlyFinish = kFind;
    __shared__ __attribute__((aligned(256))) uint32_t lut[256 * 64];
    extern __shared__ __attribute__((aligned(16))) uint8_t bufs[];   // 2 x (K tile | V^T tile)
    // Rows whose norm times a centroid would not fit fp16 are stored divided by a power of two.
    // big_tile[buf] = tile + 1 marks a tile that holds such rows; scale_exp[buf] holds the exponents,
    // K rows 0..TT-1 then V rows 0..TT-1, each tagged with tile + 1 in its upper bits (an entry with
    // another tag is left over from an earlier tile and reads as 0).
    __shared__ int big_tile[2];
    __shared__ __attribute__((aligned(16))) int scale_exp[2][128];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m32 = lane & 31, hf = lane >> 5;     // 32x32 MFMA: column (query row) and lane half
    // Workgroups reach the CUs in the order of their linear index, round after round, and under a
    // causal mask their durations grow with the query position.  Position fastest, (batch, head)
    // slow, and the position order reversed in every other round over the chip: whichever way the
    // rounds land on the CUs, each CU sees long and short workgroups alternate.
    int b, hkv, wg, piece = 0, pieces = 1;
    // What does not depend on the workgroup's work is asked for before it looks for it.  The start of a workgroup is one serial
    // chain (its work, the query rows, the rotation, the first tile); with the matrix fetched under the search, its operands
    // where the tiles will be, so that the tables are filled meanwhile, and wavefronts without a unit out of the
    // products, the first tile of one query over 4 x 2500 ring-buffer tokens begins after 6.5 us instead of 9.7 (24.3 -> 21.9 us
    // in all), 16 heads x 3001 tokens of 256 coordinates 220 -> 208 us.
    SeqShape first{};
    if constexpr (kFind && PAGED) first = lane_shape(p, 0, lane);
    const float cent_k = p.centroids_k[lane & 15], cent_v = p.centroids_v[lane & 15];
    constexpr int RROUNDS = Cfg::RROUNDS, RBLK = Cfg::RBLK;
    RotationBlocks<D> rot{p.rotation, p.rot_col_major != 0, bufs, reinterpret_cast<uint8_t*>(lut), w, lane, m32, hf, {}};
    if constexpr (kEarlyFetch) rot.fetch(false, 0);
    if constexpr (kFind) {
        // the KV heads of a place are neighbours: each XCD serves few of them
        const int at = int(blockIdx.x + gridDim.x * blockIdx.y);
        static_assert(PAGED || WORK == kAllPieces, "contiguous launches are in grid order or all in pieces");
        WorkItem it;
        if constexpr (PAGED) it = find_item<D, kSplit>(p, at, first, lane);
        else it = find_prompt_item(p, at);
        if (it.seq < 0) return;                            // the grid is sized for the most work possible
        b = it.seq; hkv = at % p.H_KV; wg = it.x; piece = it.piece; pieces = it.pieces;
    } else {
        const int lin = int(blockIdx.x) + int(gridDim.x) * (int(blockIdx.y) + int(gridDim.y) * int(blockIdx.z));
        const int pair = lin / int(gridDim.x);
        b = pair / int(gridDim.y); hkv = pair % int(gridDim.y);
        const int x_in_pair = lin % int(gridDim.x);
        // The direction is a function of the pair alone (the round its first workgroup falls in), so
        // inside a pair x -> wg is a bijection whatever the grid and the CU count are.
        const bool flip = (((int64_t(pair) * int64_t(gridDim.x)) / p.round_slots) & 1) != 0;
        wg = flip ? x_in_pair : int(gridDim.x) - 1 - x_in_pair;
    }

    // ---- this sequence -----------------------------------------------------------------------
    int NQ = p.N_Q, NKV = p.N_KV, qoff = 0;
    int64_t q_row0 = (int64_t(b) * p.H_Q) * p.N_Q;     // first row of head 0 in q / out, in rows of 128
    int q_stride = D;                                  // elements between consecutive positions of a head
    if (PAGED) {
        const int first = p.cu_seqlens_q[b];
        NQ = p.cu_seqlens_q[b + 1] - first;
        NKV = p.seq_lens[b];
        NKV = NKV < 0 ? 0 : (NKV > (p.max_blocks << p.bs_log2) ? (p.max_blocks << p.bs_log2) : NKV);
        qoff = NKV - NQ > 0 ? NKV - NQ : 0;
        q_row0 = int64_t(first) * p.H_Q;
        q_stride = p.H_Q * D;
        if (NQ <= 0) return;
    }

    // ---- units --------------------------------------------------------------------------
    const int nblk = (NQ + 31) >> 5;
    const int units = nblk * p.G;
    const int unit_raw = 8 * wg + w;
    const bool unit_live = unit_raw < units;
    const int unit = unit_live ? unit_raw : units - 1;
    const int hq = hkv * p.G + unit % p.G;
    const int pos0 = 32 * (unit / p.G);
    const int last_unit = 8 * wg + 7 < units - 1 ? 8 * wg + 7 : units - 1;
    int wg_maxpos = 32 * (last_unit / p.G) + 31;
    wg_maxpos = wg_maxpos < NQ - 1 ? wg_maxpos : NQ - 1;
    int my_maxpos = pos0 + 31 < NQ - 1 ? pos0 + 31 : NQ - 1;
    const int all_tiles = (NKV + TT - 1) >> TS;
    int ntiles = all_tiles, my_tiles = all_tiles;
    if (p.causal) {
        ntiles = ((qoff + wg_maxpos) >> TS) + 1 < all_tiles ? ((qoff + wg_maxpos) >> TS) + 1 : all_tiles;
        my_tiles = ((qoff + my_maxpos) >> TS) + 1 < all_tiles ? ((qoff + my_maxpos) >> TS) + 1 : all_tiles;
    }
    // this piece's tiles: first_tile .. ntiles - 1 (of this wavefront: .. my_tiles - 1).  Pieces are cut between the
    // schedule's tiles of 64 keys.
    int first_tile = 0;
    if (kSplit && pieces > 1) {
        constexpr int SH = 6 - TS;
        const int whole = (ntiles + (1 << SH) - 1) >> SH;
        first_tile = int(int64_t(whole) * piece / pieces) << SH;
        const int end = int(int64_t(whole) * (piece + 1) / pieces) << SH;
        ntiles = ntiles < end ? ntiles : end;
        my_tiles = my_tiles < ntiles ? my_tiles : ntiles;
    }
    if (!unit_live) my_tiles = 0;

    static_assert(2 * Cfg::RTERM <= int(sizeof(lut)) && 2 * Cfg::RTERM <= 2 * kPfBufBytes,
                  "the rotation operands fit where the tiles are, and at 256 coordinates every second round's where the tables are");
    // cleared here: the barriers of the query stage order this before the first dequantisation
    if (tid < 2) big_tile[tid] = 0;
    if (tid < 256) (&scale_exp[0][0])[tid] = 0;
    const uint8_t* lutb = reinterpret_cast<const uint8_t*>(lut);
    const uint32_t lk = 4u * (lane & 31), lv = 128u + lk;

    // ---- dequantisation plan ------------------------------------------------------------------
    const int64_t k_row0 = PAGED ? 0 : (int64_t(b) * p.H_KV + hkv) * p.k_cap;
    const int64_t v_row0 = PAGED ? 0 : (int64_t(b) * p.H_KV + hkv) * p.v_cap;
    const uint8_t* kp = p.k_packed + k_row0 * PB;
    const uint8_t* vp = p.v_packed + v_row0 * PB;
    const float* knp = p.k_norms + k_row0;
    const float* vnp = p.v_norms + v_row0;
    // Work items of the dequantisation.  K: (token of the tile, 16-coordinate group); V: (token pair, dword
    // of the packed row).  head_dim 128 and 256: 512 of each, every thread takes one of both; head_dim 64: 256
    // of each, wavefronts 0..3 take the V items and wavefronts 4..7 the K items.
    constexpr bool kSplitRoles = D == 64;
    const bool does_k = !kSplitRoles || w >= 4;
    const bool does_v = !kSplitRoles || w < 4;
    int gqk, tk, jv, tp;
    if constexpr (D == 256) {
        // as for 128, with 4 tokens x 16 groups and 4 pairs x 16 dwords a wavefront
        gqk = (lane & 3) | ((lane >> 1) & 4) | ((lane >> 2) & 8);
        tk = 4 * w + ((lane >> 2) & 1) + ((lane >> 3) & 2);
        jv = (lane & 7) | ((lane >> 2) & 8) | ((w >> 2) << 4);
        tp = 8 * ((w >> 1) & 1) + 2 * (w & 1) + ((lane >> 3) & 1) + 4 * ((lane >> 4) & 1);
    } else if constexpr (!kSplitRoles) {
        // K lane bits (g0 g1 t0 g2 t1 t2): eight consecutive lanes hold four groups of two consecutive
        // tokens, so the 128 bytes they store with one 16-byte write each fall into 32 different banks
        // (token rows are 272 bytes apart: 4 banks).
        gqk = (lane & 3) | ((lane >> 1) & 4);
        tk = 8 * w + ((lane >> 2) & 1) + ((lane >> 3) & 6);
        // V: the four pairs of a wavefront are the ones whose positions share a 16-byte group of the
        // transposed tile (0, 2, 4, 6 within it); lane bits (j0 j1 j2 p0 p1 j3): each half of the
        // wavefront holds all four pairs and eight dwords, so that its store covers all 32 banks once.
        jv = (lane & 7) | ((lane >> 2) & 8);
        tp = 8 * (w >> 1) + 2 * (w & 1) + ((lane >> 3) & 1) + 4 * ((lane >> 4) & 1);
    } else {
        // K (wavefronts 4..7): lane bits (g0 g1 t0 t1 t2 t3), 16 tokens per wavefront
        gqk = lane & 3;
        tk = 16 * (w & 3) + (lane >> 2);
        // V (wavefronts 0..3): lane bits (j0 j1 j2 p0 p1 p2): eight pairs per wavefront, the four of
        // each half sharing a 16-byte group of the transposed tile
        jv = lane & 7;
        const int i8 = lane >> 3;                       // 0..7
        tp = 8 * (w & 3) + 2 * (i8 >> 2) + (i8 & 1) + 4 * ((i8 >> 1) & 1);
    }
    const int k_wr = tk * kPfKStride + gqk * 32;
    // (256 coordinates: the registers are few, the variants of an offset are made where they are used)
    int v_wr[TT == 64 ? 8 : 1];
    {
        const int tt = 2 * tp, t16 = tt & 15;
        const int posv = (tt & ~15) + 8 * ((t16 >> 2) & 1) + 4 * ((t16 >> 3) & 1) + (t16 & 3);
        const int giv = posv >> 3, within = posv & 7;
        if constexpr (TT == 64) {
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int d = 8 * jv + k;
                const int physg = giv ^ k ^ (jv & 7);
                v_wr[k] = kPfKBytes + d * 128 + 16 * physg + 2 * within;
            }
        } else {
            v_wr[0] = kPfKBytes + jv * 512 + 16 * (giv ^ (jv & 7)) + 2 * within;
        }
    }
    // Offset of coordinate 8 jv + k.  Tiles of 32 tokens: 128 bytes hold two coordinate rows of four groups, and the
    // eight 16-byte places are permuted so that eight dwords of a store, or eight rows of an operand read, fall into eight.
    auto v_write = [&](int k) {
        if constexpr (TT == 64) {
            return v_wr[k];
        } else {
            int base = v_wr[0];
            asm volatile("" : "+v"(base));
            return (base ^ (16 * (4 * (k & 1) + (k >> 1)))) + (k >> 1) * 128;
        }
    };
    uint2v kraw = {0u, 0u};
    uint32_t vra = 0u, vrb = 0u;
    float nk = 0.0f, nv0 = 0.0f, nv1 = 0.0f;
    auto issue_loads = [&](int tile_raw) {
        const int tile = tile_raw < ntiles ? tile_raw : ntiles - 1;   // past the end: the last tile again, never used
        const int t0 = tile > 0 ? tile * TT : 0;
        const int last = NKV > 0 ? NKV - 1 : 0;
        const int tkk = t0 + tk < last ? t0 + tk : last;
        const int ta = t0 + 2 * tp < last ? t0 + 2 * tp : last;
        const int tb = t0 + 2 * tp + 1 < last ? t0 + 2 * tp + 1 : last;
        if (PAGED) {
            // token t of the sequence: row t % BS of page block_table[t / BS]; the row holds
            // [K idx H*64 | K norm H*4 | V idx H*64 | V norm H*4]
            const int H = p.H_KV;
            const int64_t row_bytes = int64_t(H) * (D + 8);
            const int32_t* bt = p.block_table + int64_t(b) * p.max_blocks;
            auto row_ptr = [&](int t) {
                int pg = bt[t >> p.bs_log2];
                pg = pg < 0 ? 0 : (pg >= p.num_blocks ? p.num_blocks - 1 : pg);
                return p.cache + ((int64_t(pg) << p.bs_log2) + (t & ((1 << p.bs_log2) - 1))) * row_bytes;
            };
            if (does_k) {
                const uint8_t* rk = row_ptr(tkk);
                kraw = *reinterpret_cast<const uint2v*>(rk + hkv * PB + 8 * gqk);
                nk = *reinterpret_cast<const float*>(rk + H * PB + 4 * hkv);
            }
            if (does_v) {
                const uint8_t* ra = row_ptr(ta);
                const uint8_t* rb2 = row_ptr(tb);
                vra = *reinterpret_cast<const uint32_t*>(ra + H * (PB + 4) + hkv * PB + 4 * jv);
                vrb = *reinterpret_cast<const uint32_t*>(rb2 + H * (PB + 4) + hkv * PB + 4 * jv);
                nv0 = *reinterpret_cast<const float*>(ra + H * (D + 4) + 4 * hkv);
                nv1 = *reinterpret_cast<const float*>(rb2 + H * (D + 4) + 4 * hkv);
            }
        } else {
            // (32-bit offsets from the wave-uniform slab pointers: a slab of 2^31 / PB tokens is far beyond
            // any context)
            if (does_k) {
                kraw = *reinterpret_cast<const uint2v*>(kp + (uint32_t(tkk) * uint32_t(PB) + 8u * uint32_t(gqk)));
                nk = knp[uint32_t(tkk)];
            }
            if (does_v) {
                vra = *reinterpret_cast<const uint32_t*>(vp + (uint32_t(ta) * uint32_t(PB) + 4u * uint32_t(jv)));
                vrb = *reinterpret_cast<const uint32_t*>(vp + (uint32_t(tb) * uint32_t(PB) + 4u * uint32_t(jv)));
                nv0 = vnp[uint32_t(ta)];
                nv1 = vnp[uint32_t(tb)];
            }
        }
    };
    auto dequant = [&](int buf, int tile) {
        uint8_t* dst = bufs + buf * kPfBufBytes;
        if (__any(__builtin_fmaxf(__builtin_fabsf(nk), __builtin_fmaxf(__builtin_fabsf(nv0), __builtin_fabsf(nv1))) >= 32768.0f)) {
            const int ek = norm_excess(nk), ev0 = norm_excess(nv0), ev1 = norm_excess(nv1);
            nk = __builtin_ldexpf(nk, -ek);
            nv0 = __builtin_ldexpf(nv0, -ev0);
            nv1 = __builtin_ldexpf(nv1, -ev1);
            const int tag = (tile + 1) << 8;
            if (does_k && gqk == 0) scale_exp[buf][tk] = tag | ek;
            if (does_v && jv == 0) {
                scale_exp[buf][TT + 2 * tp] = tag | ev0;
                scale_exp[buf][TT + 2 * tp + 1] = tag | ev1;
            }
            if ((ek | ev0 | ev1) != 0) big_tile[buf] = tile + 1;
        }
        if (does_k) {      // uniform over the wavefront
            const _Float16 hk = _Float16(nk);
            const half2v nk2 = {hk, hk};
            const uint4v a0 = lookup_word(lutb, kraw.x, lk);   // coordinates 0..7 of the group
            const uint4v a1 = lookup_word(lutb, kraw.y, lk);   // coordinates 8..15
            // positions 0..7 = coordinates (0..3, 8..11), positions 8..15 = (4..7, 12..15)
            const uint4v w0 = {scale_pair(a0.x, nk2), scale_pair(a0.y, nk2), scale_pair(a1.x, nk2), scale_pair(a1.y, nk2)};
            const uint4v w1 = {scale_pair(a0.z, nk2), scale_pair(a0.w, nk2), scale_pair(a1.z, nk2), scale_pair(a1.w, nk2)};
            *reinterpret_cast<uint4v*>(dst + k_wr) = w0;
            *reinterpret_cast<uint4v*>(dst + k_wr + 16) = w1;
        }
        if (does_v) {
            // V: 2x2 nibble transpose, so that a byte holds one coordinate of the two tokens
            const uint32_t X = (vra & 0xF0F0F0F0u) | ((vrb >> 4) & 0x0F0F0F0Fu);   // even coordinates
            const uint32_t Y = ((vra << 4) & 0xF0F0F0F0u) | (vrb & 0x0F0F0F0Fu);   // odd coordinates
            const half2v nv2 = {_Float16(nv0), _Float16(nv1)};
            const uint4v xe = lookup_word(lutb, X, lv);
            const uint4v yo = lookup_word(lutb, Y, lv);
            const uint32_t xs[4] = {xe.x, xe.y, xe.z, xe.w}, ys[4] = {yo.x, yo.y, yo.z, yo.w};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                *reinterpret_cast<uint32_t*>(dst + v_write(2 * c)) = scale_pair(xs[c], nv2);
                *reinterpret_cast<uint32_t*>(dst + v_write(2 * c + 1)) = scale_pair(ys[c], nv2);
            }
        }
    };

    // ---- query: rotate this wavefront's 32 rows, round to the query dtype, scale to fp16 ----------
    half8 qb[NKS];
    float krow = 0.0f;
    {
        const uint16_t* qbase = PAGED ? p.q + (q_row0 + hq) * D : p.q + (q_row0 + int64_t(hq) * NQ) * D;
        const int pos = pos0 + m32 < NQ ? pos0 + m32 : NQ - 1;
        uint4v raw[NKS];
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
            raw[ks] = *reinterpret_cast<const uint4v*>(qbase + int64_t(pos) * q_stride + 16 * ks + 8 * hf);
        if constexpr (!kEarlyFetch) rot.fetch(false, 0);
        issue_loads(first_tile);
        // The matrix lies where the tiles will be, so the tables are there before the products begin; at 256 coordinates they
        // take turns with the rounds of the matrix and are filled under the last one.
        if (RROUNDS == 1) fill_pair_tables<8>(lut, cent_k, cent_v, 15, w, lane);
        rot.put(0);
        if (RROUNDS > 1) rot.fetch(false, 1);
        // the rows are exact in fp16 up to a power of two
        half8 qa[NKS];
        float mx = 0.0f;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                mx = __builtin_fmaxf(mx, __builtin_fmaxf(__builtin_fabsf(load_elem<DT>(uint16_t(raw[ks][i] & 0xffffu))),
                                                         __builtin_fabsf(load_elem<DT>(uint16_t(raw[ks][i] >> 16)))));
        const int ex = row_exponent(mx);
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                qa[ks][2 * i] = _Float16(load_elem<DT>(uint16_t(raw[ks][i] & 0xffffu)) * pow2(-ex));
                qa[ks][2 * i + 1] = _Float16(load_elem<DT>(uint16_t(raw[ks][i] >> 16)) * pow2(-ex));
            }
        float16v rows[D == 256 ? 1 : NOB] = {};
        uint32_t rows16[D == 256 ? NOB : 1][8] = {};     // 256 coordinates: held as the 16-bit pairs they are rounded to
        float mr = 0.0f;
        // A wavefront without a unit leaves the LDS and the matrix cores to the others: half of them where one query of four
        // heads shares its keys.  In the forms without pieces the branch is opaque: the compiler took it for a reason to hold
        // two copies of the tile loop (64 coordinates 193 registers instead of 170, 40 queries over 100 to 4000 keys 88.0 and
        // 83.9 us, 85.2 before there was a branch; 16 x 300 tokens of 128, grid order, 106 scalar registers and 5 spilled instead of
        // 65).  With pieces it does not, and opaque costs 1 % (mixed batch of 12 at 64 coordinates 266 and 270 us).
        int live = 1;
        if constexpr (kSkipDead && WORK != kPieces) {
            live = __builtin_amdgcn_readfirstlane(unit_live ? 1 : 0);
            asm volatile("" : "+s"(live));
        }
#pragma unroll
        for (int round = 0; round < RROUNDS; ++round) {
            __syncthreads();                            // this round's operands are there, the ones before are done with
            if (round + 1 < RROUNDS) rot.put(round + 1);
            if (round + 2 < RROUNDS) rot.fetch(false, round + 2);
            if (RROUNDS > 1 && round == RROUNDS - 1) fill_pair_tables<8>(lut, cent_k, cent_v, 15, w, lane);
            if constexpr (WORK == kPieces) {
                if (!unit_live) continue;
            } else if constexpr (kSkipDead) {
                if (live == 0) continue;
            }
            rot.template products<false>(round, qa, qa, [&](int jr, const float16v& hi, const float16v& lo) {
                const int jb = RBLK * round + jr;
                if constexpr (D == 256) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const uint16_t x = store_elem<DT>((hi[2 * i] + lo[2 * i] * (1.0f / 4096.0f)) * pow2(ex));
                        const uint16_t y = store_elem<DT>((hi[2 * i + 1] + lo[2 * i + 1] * (1.0f / 4096.0f)) * pow2(ex));
                        mr = __builtin_fmaxf(mr, __builtin_fmaxf(__builtin_fabsf(load_elem<DT>(x)), __builtin_fabsf(load_elem<DT>(y))));
                        rows16[jb][i] = uint32_t(x) | uint32_t(y) << 16;
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        rows[jb][r] = load_elem<DT>(store_elem<DT>((hi[r] + lo[r] * (1.0f / 4096.0f)) * pow2(ex)));
                        mr = __builtin_fmaxf(mr, __builtin_fabsf(rows[jb][r]));
                    }
                }
            });
        }
        const int er = row_exponent(mr);
        krow = p.scale_log2e * pow2(er);
        // the result registers 8 u .. 8 u + 7 of a block are the operand of k-step u (the order of the K tile)
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float v;
                if constexpr (D == 256) v = load_elem<DT>(uint16_t(rows16[ks >> 1][4 * (ks & 1) + (e >> 1)] >> (16 * (e & 1))));
                else v = rows[ks >> 1][8 * (ks & 1) + e];
                qb[ks][e] = _Float16(v * pow2(-er));
            }
        __syncthreads();   // the rotation operands become tiles
    }

    // ---- lane-constant LDS read offsets ----------------------------------------------------------
    const int k_rd = m32 * kPfKStride + 16 * hf;
    int v_rd[TT == 64 ? 8 : 1];
    {
        const int lanex = TT == 64 ? hf ^ (m32 & 7) ^ (m32 >> 3) : hf ^ (4 * (m32 & 1) + ((m32 >> 1) & 3)) ^ (m32 >> 3);
#pragma unroll
        for (int c = 0; c < (TT == 64 ? 8 : 1); ++c) v_rd[c] = kPfKBytes + (TT == 64 ? m32 : m32 >> 1) * 128 + 16 * (lanex ^ c);
    }

    // ---- running state -----------------------------------------------------------------------------
    float16v O[NOB];
#pragma unroll
    for (int ob = 0; ob < NOB; ++ob)
#pragma unroll
        for (int r = 0; r < 16; ++r) O[ob][r] = 0.0f;
    float m_run = -__builtin_inff();
    float l_run = 0.0f;
    const int qpos = qoff + pos0 + m32;            // position among the keys

    auto compute = [&](int tile, int buf) {
        const uint8_t* kt = bufs + buf * kPfBufBytes;
        float16v S[NTB];
#pragma unroll
        for (int tb = 0; tb < NTB; ++tb) {
#pragma unroll
            for (int r = 0; r < 16; ++r) S[tb][r] = 0.0f;
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                const half8 a = *reinterpret_cast<const half8*>(kt + k_rd + 32 * tb * kPfKStride + 32 * ks);
                S[tb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qb[ks], S[tb], 0, 0, 0);
            }
        }
        const int t0 = tile * TT;
        // rows stored divided by a power of two (norms beyond fp16's range): wavefront-uniform, rare
        const bool big = __builtin_amdgcn_readfirstlane(big_tile[buf]) == tile + 1;
        auto exps_of = [&](int first) {        // the exponents of four consecutive rows of this tile
            const int4v raw = *reinterpret_cast<const int4v*>(&scale_exp[buf][first]);
            int4v e;
#pragma unroll
            for (int c = 0; c < 4; ++c) e[c] = (raw[c] >> 8) == tile + 1 ? (raw[c] & 0xff) : 0;
            return e;
        };
        if (big) {
#pragma unroll
            for (int tb = 0; tb < NTB; ++tb)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int4v e = exps_of(32 * tb + 8 * q + 4 * hf);
#pragma unroll
                    for (int c = 0; c < 4; ++c) S[tb][4 * q + c] = __builtin_ldexpf(S[tb][4 * q + c], e[c]);
                }
        }
        const bool need_mask = (t0 + TT - 1 >= NKV) || (p.causal && t0 + TT - 1 > qoff + pos0);   // wavefront-uniform
        if (need_mask) {
            int lim = NKV - 1;
            if (p.causal && qpos < lim) lim = qpos;
            lim -= t0;                         // token offsets <= lim are visible
#pragma unroll
            for (int tb = 0; tb < NTB; ++tb)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int off = 32 * tb + 8 * (r >> 2) + 4 * hf + (r & 3);
                    if (off > lim) S[tb][r] = -__builtin_inff();
                }
        }
        float cand;
        if (!big) {
            float mx = S[0][0];
#pragma unroll
            for (int tb = 0; tb < NTB; ++tb)
#pragma unroll
                for (int r = 0; r < 16; ++r) mx = __builtin_fmaxf(mx, S[tb][r]);
            cand = mx * krow;
        } else {
            // a value row stored divided by 2^e gets its weight multiplied by 2^e: the reference is
            // taken over score + e, so that these weights stay below 16 as well
            cand = -__builtin_inff();
#pragma unroll
            for (int tb = 0; tb < NTB; ++tb)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int4v e = exps_of(TT + 32 * tb + 8 * q + 4 * hf);
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        cand = __builtin_fmaxf(cand, __builtin_fmaf(S[tb][4 * q + c], krow, float(e[c])));
                }
        }
        cand = max_xor32(cand);
        // the running maximum moves only when it would grow by more than 2^4: the weights stay
        // below 16 and the rescale of the accumulator registers becomes rare.  At 256 coordinates it always moves, so
        // that the largest weight is exactly 1, as on the general kernel: error against 64 bits 8.88e-4 (8.92e-4
        // otherwise, 8.88e-4 there; fp16, 3001 tokens) for 5 % of the time.
        const float mnew = cand > m_run + (D == 256 ? 0.0f : 4.0f) ? cand : m_run;
        const float ms = mnew == -__builtin_inff() ? 0.0f : mnew;
        const float alpha = __builtin_amdgcn_exp2f(m_run - ms);
        m_run = mnew;
        uint4v pbv[NVS];
        float ps = 0.0f;
        // two copies of the weight loop, so that the common one has no branch inside (the values of a
        // loop with a rare branch in it are copied where the paths meet)
        if (!big) {
            const half2v ones = {_Float16(1.0f), _Float16(1.0f)};
#pragma unroll
            for (int s = 0; s < NVS; ++s) {
                float pe[8];
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    pe[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(S[s >> 1][8 * (s & 1) + e], krow, -ms));
                const uint32_t pw[4] = {pack_weights<D>(pe[0], pe[1]), pack_weights<D>(pe[2], pe[3]), pack_weights<D>(pe[4], pe[5]), pack_weights<D>(pe[6], pe[7])};
                // the denominator sums the weights as the second product sees them (fp16, one
                // v_dot2_f32_f16 per pair)
#pragma unroll
                for (int c = 0; c < 4; ++c) ps = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2v, pw[c]), ones, ps, false);
                pbv[s] = uint4v{pw[0], pw[1], pw[2], pw[3]};
            }
        } else {
#pragma unroll
            for (int s = 0; s < NVS; ++s) {
                float pe[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    pe[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(S[s >> 1][8 * (s & 1) + e], krow, -ms));
                    ps += pe[e];
                }
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const int4v ev = exps_of(TT + 32 * (s >> 1) + 8 * (2 * (s & 1) + q) + 4 * hf);
#pragma unroll
                    for (int c = 0; c < 4; ++c) pe[4 * q + c] = __builtin_ldexpf(pe[4 * q + c], ev[c]);
                }
                pbv[s] = uint4v{pack_weights<D>(pe[0], pe[1]), pack_weights<D>(pe[2], pe[3]), pack_weights<D>(pe[4], pe[5]), pack_weights<D>(pe[6], pe[7])};
            }
        }
        l_run = __builtin_fmaf(l_run, alpha, ps);
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int ob = 0; ob < NOB; ++ob)
#pragma unroll
                for (int r = 0; r < 16; ++r) O[ob][r] *= alpha;
        }
        // The V operands of 16 tokens (one per 32-coordinate block) are read two such groups ahead of
        // the products that use them (the compiler on its own reads one product ahead, which does
        // not cover the LDS round trip): fences keep the groups in this order.
        auto v_operand = [&](int ob, int s) {
            const int c = (2 * s) ^ (4 * (ob & 1));
            if constexpr (TT == 64) {
                return *reinterpret_cast<const half8*>(kt + v_rd[c] + ob * (64 * TT));
            } else {
                int base = v_rd[0];
                asm volatile("" : "+v"(base));
                return *reinterpret_cast<const half8*>(kt + (base ^ (16 * c)) + ob * (64 * TT));
            }
        };
        // groups of VG blocks; at 256 coordinates the registers allow two blocks (of the eight) a group
        constexpr int VG = D == 256 ? 2 : NOB, NG = NVS * NOB / VG;
        half8 va[NG][VG];
        auto read_group = [&](int g) {
#pragma unroll
            for (int k = 0; k < VG; ++k) va[g][k] = v_operand((g * VG) % NOB + k, (g * VG) / NOB);
        };
        read_group(0);
        read_group(1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            if (g + 2 < NG) {
                read_group(g + 2);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int k = 0; k < VG; ++k) {
                const int ob = (g * VG) % NOB + k;
                O[ob] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[g][k], __builtin_bit_cast(half8, pbv[(g * VG) / NOB]), O[ob], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // ---- tiles ----------------------------------------------------------------------------------------
    dequant(first_tile & 1, first_tile);
    // (at 256 coordinates the scheduler drew the first tile's end into the loop of this form: one prompt of 8192 tokens, 16 heads
    // over 4, 962 us without the fence and 951 with it, 4 prompts of 4096 1031 and 1026)
    if constexpr (D == 256 && WORK == kOrdered) __builtin_amdgcn_sched_barrier(0);
    issue_loads(first_tile + 1);
    // The dequantisation of tile i + 1 and the products of tile i sit in one basic block (no
    // conditions between them), so that the lookups and LDS writes of the one interleave with
    // the MFMAs of the other.
    int i = first_tile;
    for (; i < my_tiles; ++i) {
        __syncthreads();                       // tile i is complete; the other buffer is free
        dequant((i + 1) & 1, i + 1);
        issue_loads(i + 2);
        compute(i, i & 1);
    }
    for (; i < ntiles; ++i) {                  // tiles only the other wavefronts of the workgroup need
        __syncthreads();
        dequant((i + 1) & 1, i + 1);
        issue_loads(i + 2);
    }

    // ---- a piece of a workgroup's keys: the rows as they are, for the combine launch ------------------------
    // Only rows that hold a query: a unit of one query left 31 rows of padding, 64 KB a piece at 4 heads of 128 (one query
    // over 4 x 2500 tokens of a ring buffer 33.5 -> 30.2 us).
    if (WORK == kAllPieces || (WORK == kPieces && pieces > 1)) {
        const float l_piece = l_run + xor_shuffle(l_run, 32);
        if (!unit_live || pos0 + m32 >= NQ) return;
        const int64_t slot = ((int64_t(b) * p.H_KV + hkv) * p.split_w + wg) * p.max_pieces + piece;
        float* dst = p.part + slot * Cfg::SLOT + w * (32 * D + 64);
#pragma unroll
        for (int ob = 0; ob < NOB; ++ob)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<float4v*>(dst + m32 * D + 32 * ob + 8 * q + 4 * hf) =
                    float4v{O[ob][4 * q], O[ob][4 * q + 1], O[ob][4 * q + 2], O[ob][4 * q + 3]};
        dst[32 * D + lane] = hf == 0 ? m_run : l_piece;
        return;
    }

    // ---- normalise, rotate back, store -------------------------------------------------------------------
    if constexpr (WORK != kAllPieces) {
        const float l_tot = l_run + xor_shuffle(l_run, 32);
        const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
        rot.fetch(true, 0);
        __syncthreads();                // every wavefront is done with the tiles and the tables
        rot.put(0);
        __syncthreads();
        finish_rows<D, DT, PAGED, kEarlyFinish>(p, rot, O, inv, unit_live, pos0, hq, NQ, q_row0, q_stride);
    }
}

// Rows of the workgroups that ran in pieces: the pieces' rows weighted by 2^(m - max m), summed and normalised, rounded
// as the kernel above rounds, rotated back.  A workgroup takes `rows` (4 or 16) rows, of one unit or (one or two queries) a few of each
// of 2^`units_log2` units, a wavefront a row at a time; blockIdx.x numbers the (sequence, KV head, workgroup) triples that may have
// been split, blockIdx.y their row groups.  With KS > 1 the columns of a row group are shared by the workgroups of blockIdx.z,
// each gathering the rows for itself, and a block of 16 columns by KS wavefronts, each 1 / KS of the contraction.
// Bound by the launch, two round trips (partials and matrix are asked for together) and the part of the matrix that a
// workgroup takes: 128 rows of 128 coordinates 5.2 us with a workgroup a row, 3.5 with four for four.
template <int D, int DT, bool PAGED, int KS>
__global__ __launch_bounds__(256) void attention_combine_kernel(const PrefillParams p, int rows, int units_log2) {
    using Cfg = PrefillCfg<D>;
    const int usplit = KS == 1 ? 0 : units_log2;
    constexpr int CBW = KS == 1 ? D / 64 : 1, CPL = D / 64;     // column blocks per wavefront, coordinates per lane
    constexpr int J = D / 32 / KS;                              // runs of 32 contraction indices per wavefront
    static_assert(J * KS == D / 32, "whole runs");
    __shared__ __attribute__((aligned(16))) float os[16 * (D + 4)];
    __shared__ float sums[KS == 1 ? 1 : 4][16][16];             // sums of the wavefronts that share a contraction
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n16 = lane & 15, g4 = lane >> 4;
    const int x = int(blockIdx.x) % p.split_w, pair = int(blockIdx.x) / p.split_w;
    const int b = pair / p.H_KV, hkv = pair % p.H_KV;
    const int pieces = PAGED ? p.left[blockIdx.x] : p.max_pieces;
    if (pieces == 0) return;
    const SeqShape sh = seq_shape<PAGED>(p, b);
    const int groups = int(gridDim.y) > (8 >> usplit) ? 2 : 1;
    const int u0 = (int(blockIdx.y) / groups) << usplit, row0 = int(blockIdx.y) % groups * rows;
    if (8 * x + u0 >= sh.units) return;
    const int rsh = (rows == 16 ? 4 : 2) - usplit;              // 2^rsh rows of a unit
    // units beside each other are heads of the same 32 positions (where there are several here, a head has only one)
    const int block = (8 * x + u0) / p.G, head0 = 8 * x + u0 - block * p.G;
    auto head_of = [&](int r) { return KS == 1 ? head0 : head0 + (r >> rsh); };
    auto row_of = [&](int r) { return KS == 1 ? row0 + r : row0 + (r & ((1 << rsh) - 1)); };             // among the unit's 32
    auto pos_of = [&](int r) { return 32 * block + row_of(r); };
    auto live = [&](int r) { return (KS == 1 || (u0 + (r >> rsh) < 8 && head_of(r) < p.G)) && pos_of(r) < sh.NQ; };
    if (!live(0)) return;

    const float* src = p.part + (int64_t(blockIdx.x) * p.max_pieces) * Cfg::SLOT;
    constexpr bool kAhead = CBW * J <= 8;         // (256 coordinates in one workgroup: too many registers)
    const int cb0 = KS == 1 ? wave : 4 / KS * int(blockIdx.z) + wave / KS, k0 = wave % KS * (D / KS);
    float rbv[kAhead ? CBW : 1][J][8];
#pragma unroll
    for (int i = 0; i < (kAhead ? CBW : 0); ++i)
        load_rotation_any<D, J>(p.rotation, p.rot_col_major != 0, false, 16 * (cb0 + 4 * i), n16, g4, rbv[i], k0);
    for (int r = wave; r < rows; r += 4) {
        if (!live(r)) {                                         // no query: the pieces left no such row
#pragma unroll
            for (int e = 0; e < CPL; ++e) os[r * (D + 4) + CPL * lane + e] = 0.0f;
            continue;
        }
        const float* unit_src = src + (KS == 1 ? u0 : u0 + (r >> rsh)) * (32 * D + 64);
        const float* head = unit_src + 32 * D + row_of(r);
        const bool have = lane < pieces;                        // (at most 32 pieces)
        const float m = have ? head[int64_t(lane) * Cfg::SLOT] : -__builtin_inff();
        const float l = have ? head[int64_t(lane) * Cfg::SLOT + 32] : 0.0f;
        const float top = wave_max(m);
        const float wgt = piece_weight(m, l, top);
        float den = 0.0f, num[CPL];
#pragma unroll
        for (int e = 0; e < CPL; ++e) num[e] = 0.0f;
        auto of_lane = [](float v, int k) { return bits_to_float(uint32_t(__builtin_amdgcn_readlane(int(float_to_bits(v)), k))); };
        for (int k0 = 0; k0 < pieces; k0 += 8) {
            float at[8][CPL];
#pragma unroll
            for (int i = 0; i < 8; ++i) {                       // eight pieces in flight (past the end: the last one again)
                const int k = k0 + i < pieces ? k0 + i : pieces - 1;
                const float* row = unit_src + int64_t(k) * Cfg::SLOT + row_of(r) * D + CPL * lane;
#pragma unroll
                for (int e = 0; e < CPL; ++e) at[i][e] = row[e];
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float wk = of_lane(wgt, k0 + i);          // (past the end 0: the last piece's row again adds nothing)
                den = __builtin_fmaf(of_lane(l, k0 + i), wk, den);
#pragma unroll
                for (int e = 0; e < CPL; ++e) num[e] = __builtin_fmaf(at[i][e], wk, num[e]);
            }
        }
        const float inv = inverse_sum(den);
#pragma unroll
        for (int e = 0; e < CPL; ++e) {
            const float v = num[e] * inv;
            os[r * (D + 4) + CPL * lane + e] = PAGED ? load_elem<DT>(store_elem<DT>(v)) : v;
        }
    }
    __syncthreads();
    float a[J][8];
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float4v v = *reinterpret_cast<const float4v*>(os + (n16 & (rows - 1)) * (D + 4) + k0 + 32 * j + 8 * g4 + 4 * h);
#pragma unroll
            for (int e = 0; e < 4; ++e) a[j][4 * h + e] = v[e];
        }
    // fp16 terms as in finish_rows, scaled row by row (the rows of a block may differ by any factor): lanes n16 + 16 g hold
    // row n16
    constexpr int kUp = PAGED ? 14 : 0;
    half8 ahi[J], alo[J];
    float mx = 0.0f;
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) mx = __builtin_fmaxf(mx, __builtin_fabsf(a[j][e]));
    const int ex = row_exponent(max_xor16(mx)) - kUp;
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const float a0 = a[j][e] * pow2(-ex), a1 = a[j][e + 1] * pow2(-ex);
            if (PAGED) {
                ahi[j][e] = _Float16(a0); ahi[j][e + 1] = _Float16(a1);
            } else {
                const auto h2 = __builtin_amdgcn_cvt_pkrtz(a0, a1);
                const auto l2 = __builtin_amdgcn_cvt_pkrtz((a0 - float(h2[0])) * 4096.0f, (a1 - float(h2[1])) * 4096.0f);
                ahi[j][e] = h2[0]; ahi[j][e + 1] = h2[1];
                alo[j][e] = l2[0]; alo[j][e + 1] = l2[1];
            }
        }
    float up[4];                       // of the result rows 4 g4 + k
#pragma unroll
    for (int k = 0; k < 4; ++k) up[k] = pow2(__shfl(ex, 4 * g4 + k, kWave));
    const int stride = PAGED ? p.H_Q * D : D, head_stride = PAGED ? D : sh.NQ * D;
    uint16_t* out = p.out + (PAGED ? int64_t(p.cu_seqlens_q[b]) : int64_t(b) * sh.NQ) * p.H_Q * D + int64_t(hkv * p.G) * head_stride;
    auto store = [&](int r, int col, float v) {
        out[int64_t(head_of(r)) * head_stride + int64_t(pos_of(r)) * stride + col] = store_elem<DT>(v);
    };
#pragma unroll
    for (int i = 0; i < CBW; ++i) {
        half8 rhi[J], rlo[J];
        if (!kAhead) load_rotation_any<D, J>(p.rotation, p.rot_col_major != 0, false, 16 * (cb0 + 4 * i), n16, g4, rbv[0], k0);
        split_rotation_block<32 * J>(rbv[kAhead ? i : 0], rhi, rlo);
        const float4v acc = PAGED ? rotate_block_f16<32 * J>(ahi, rhi, rlo) : rotate_block_f16x3<32 * J>(ahi, alo, rhi, rlo);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int r = 4 * g4 + k;
            if constexpr (KS > 1) sums[wave][r][n16] = acc[k] * up[k];
            else if (r < rows && live(r)) store(r, 16 * (cb0 + 4 * i) + n16, acc[k] * up[k]);
        }
    }
    if constexpr (KS > 1) {
        __syncthreads();
        for (int c = threadIdx.x; c < 4 / KS * 16 * rows; c += 256) {
            const int col = c & 15, r = (c >> 4) & (rows - 1), cb = (c >> 4) / rows;
            float sum = sums[cb * KS][r][col];
#pragma unroll
            for (int k = 1; k < KS; ++k) sum += sums[cb * KS + k][r][col];
            if (live(r)) store(r, 16 * (4 / KS * int(blockIdx.z) + cb) + col, sum);
        }
    }
}

// The same for whole prompts in pieces, where the rotation is the work: a workgroup as the one that left the pieces, its
// wavefronts gather their 32 rows in the accumulators and end as that kernel does (the kernel above fetches and splits the
// matrix for every 16 rows).  When it was added, 16 heads x 3001 tokens of 256 coordinates, 188 workgroups in two pieces: 298 us
// with the kernel above, 240 with this one (203 later; where the caller gives room for expanded
// keys and values, 136 without either); 8 heads x 5000 tokens of 128, 157 workgroups: 140 and 121; 16 heads x
// 2000 tokens of 64, 128 workgroups: 54.6 and 48.3 (45.8 later).  With 63 workgroups in four pieces the smaller workgroups above
// are faster (128 and 148 us at 256 coordinates, 55 and 68 at 128): this one runs from half a round of workgroups on.  At 256
// coordinates the rounds of the matrix share one area (64 KB, so that two workgroups fit a CU): with two of them 14 registers
// were spilled and 16 heads x 3001 tokens took 209 us, 202 with one.
template <int D, int DT, bool PAGED>
__global__ __launch_bounds__(512) void attention_combine_prompts_kernel(const PrefillParams p) {
    using Cfg = PrefillCfg<D>;
    constexpr int NOB = Cfg::NOB;
    __shared__ __attribute__((aligned(16))) uint8_t share[2 * Cfg::RTERM];
    const int tid = threadIdx.x, lane = tid & 63, m32 = lane & 31, hf = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wg = int(blockIdx.x) % p.split_w, pair = int(blockIdx.x) / p.split_w;
    const int b = pair / p.H_KV, hkv = pair % p.H_KV;
    const int pieces = PAGED ? p.left[blockIdx.x] : p.max_pieces;
    if (pieces == 0) return;
    const SeqShape sh = seq_shape<PAGED>(p, b);
    RotationBlocks<D, 1> rot{p.rotation, p.rot_col_major != 0, share, nullptr, w, lane, m32, hf, {}};
    rot.fetch(true, 0);

    const bool unit_live = 8 * wg + w < sh.units;              // a dead unit left no rows
    const int unit = unit_live ? 8 * wg + w : sh.units - 1;
    const int hq = hkv * p.G + unit % p.G, pos0 = 32 * (unit / p.G);
    float16v O[NOB];
#pragma unroll
    for (int ob = 0; ob < NOB; ++ob)
#pragma unroll
        for (int r = 0; r < 16; ++r) O[ob][r] = 0.0f;
    float den = 0.0f;
    if (unit_live && pos0 + m32 < sh.NQ) {                     // no other rows were left
        const float* src = p.part + int64_t(blockIdx.x) * p.max_pieces * Cfg::SLOT + w * (32 * D + 64);
        float top = -__builtin_inff();
        for (int k = 0; k < pieces; ++k) top = __builtin_fmaxf(top, src[int64_t(k) * Cfg::SLOT + 32 * D + m32]);
        for (int k = 0; k < pieces; ++k) {
            const float* slot = src + int64_t(k) * Cfg::SLOT;
            const float m = slot[32 * D + m32], l = slot[32 * D + 32 + m32];
            const float wk = piece_weight(m, l, top);
            den = __builtin_fmaf(l, wk, den);
#pragma unroll
            for (int ob = 0; ob < NOB; ++ob)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4v v = *reinterpret_cast<const float4v*>(slot + m32 * D + 32 * ob + 8 * q + 4 * hf);
#pragma unroll
                    for (int c = 0; c < 4; ++c) O[ob][4 * q + c] = __builtin_fmaf(v[c], wk, O[ob][4 * q + c]);
                }
        }
    }
    rot.put(0);
    __syncthreads();
    const int64_t q_row0 = PAGED ? int64_t(p.cu_seqlens_q[b]) * p.H_Q : int64_t(b) * p.H_Q * p.N_Q;
    finish_rows<D, DT, PAGED, true>(p, rot, O, inverse_sum(den), unit_live, pos0, hq, sh.NQ, q_row0,
                              PAGED ? p.H_Q * D : D);
}

template <int D, int DT, bool PAGED, int WORK>
int launch_prefill_as(const PrefillParams& p, dim3 grid, int max_q, hipStream_t s) {
    const size_t lds = 2 * size_t(PrefillCfg<D>::BUF);
    auto kern = fused_tq_attention_kernel<D, DT, PAGED, WORK>;
    if (!fq_host::lds_limit_raised(reinterpret_cast<const void*>(kern), lds)) return FQ_ERR_LAUNCH;
    hipLaunchKernelGGL(kern, grid, dim3(512), lds, s, p);
    const int st = fq_host::check_launch();
    if constexpr (WORK == kPieces || WORK == kAllPieces) {
        if (st != FQ_OK) return st;
        const int64_t slots = int64_t(p.num_seqs) * p.H_KV * p.split_w;
        if (p.split_w > 1 && 2 * slots >= p.round_slots) {
            hipLaunchKernelGGL((attention_combine_prompts_kernel<D, DT, PAGED>), dim3(unsigned(slots)), dim3(512), 0, s, p);
            return fq_host::check_launch();
        }
        const int rows = max_q <= 4 ? 4 : 16;
        const int groups = max_q <= 16 ? 1 : 2;             // 32 rows a unit at most
        // Workgroups share the columns of the rows while CUs are idle, at 256 coordinates up to two workgroups a CU.  One query
        // over ring buffers, 32 heads over 8 of 128, bf16, in us, without and with: 4 x 2500 tokens 21.8, 20.2; 1 x 16,000 27.9, 26.3;
        // 16 x 700 (512 workgroups) 27.3, 27.4; 5 queries over 4 x 2500 (512) 23.0, 24.3.  16 heads over 4 of 256: 2 x 1000 42.1, 35.6;
        // 8 x 1500 (512) 42.9, 38.7; 2 queries over 8 x 1000, 32 heads over 8 (2048), 43.8, 44.4.  At 64 coordinates, where
        // the matrix is 16 KB, nothing helps: 15.1 and 15.3.
        if constexpr (D >= 128) {
            constexpr int KS = D == 256 ? 4 : 2, CS = D / 64 * KS;
            const int usplit = max_q <= 1 ? 2 : (max_q == 2 ? 1 : 0);
            const int units = p.G * ((max_q + 31) / 32) < 8 ? p.G * ((max_q + 31) / 32) : 8;
            const int64_t live = slots * ((units + (1 << usplit) - 1) >> usplit) * groups * CS;
            const bool shared = live <= (D == 256 ? 2 : 1) * int64_t(p.round_slots);
            if (shared) {
                hipLaunchKernelGGL((attention_combine_kernel<D, DT, PAGED, KS>), dim3(unsigned(slots), (8 >> usplit) * groups, CS), dim3(256),
                                   0, s, p, rows, usplit);
                return fq_host::check_launch();
            }
        }
        hipLaunchKernelGGL((attention_combine_kernel<D, DT, PAGED, 1>), dim3(unsigned(slots), 8 * groups), dim3(256), 0, s, p, rows, 0);
        return fq_host::check_launch();
    }
    return st;
}

template <int D, bool PAGED, int WORK>
int launch_prefill_dtype(const PrefillParams& p, dim3 grid, int max_q, int dtype, hipStream_t s) {
    return dtype == FQ_F16 ? launch_prefill_as<D, FQ_F16, PAGED, WORK>(p, grid, max_q, s)
                           : launch_prefill_as<D, FQ_BF16, PAGED, WORK>(p, grid, max_q, s);
}

// The forms that are built: contiguous launches are all in pieces or not at all; of the paged ones a batch whose every
// workgroup has a place in `part` leaves all rows there at 256 coordinates (Work says why).
template <int D, bool PAGED>
int launch_prefill_dim(PrefillParams& p, dim3 grid, int max_q, int dtype, hipStream_t s) {
    p.all_in_part = p.max_pieces > 1 && (!PAGED || (D == 256 && p.split_w == p.max_w));
    if (p.all_in_part) {
        if constexpr (!PAGED || D == 256) return launch_prefill_dtype<D, PAGED, kAllPieces>(p, grid, max_q, dtype, s);
    }
    if constexpr (!PAGED) {
        return launch_prefill_dtype<D, PAGED, kGrid>(p, grid, max_q, dtype, s);
    } else {
        if (p.max_pieces > 1) return launch_prefill_dtype<D, PAGED, kPieces>(p, grid, max_q, dtype, s);
        return launch_prefill_dtype<D, PAGED, kOrdered>(p, grid, max_q, dtype, s);
    }
}

template <bool PAGED>
int launch_prefill(PrefillParams& p, int D, dim3 grid, int max_q, int dtype, hipStream_t s) {
    if (D == 64) return launch_prefill_dim<64, PAGED>(p, grid, max_q, dtype, s);
    if (D == 256) return launch_prefill_dim<256, PAGED>(p, grid, max_q, dtype, s);
    return launch_prefill_dim<128, PAGED>(p, grid, max_q, dtype, s);
}

// n workgroups in rows of at most 2^20 (a grid row holds fewer than 2^32 threads); the last row's surplus finds no work.
inline dim3 folded_grid(int64_t n) {
    const int64_t x = n < (1 << 20) ? n : (1 << 20);
    return dim3(unsigned(x), unsigned((n + x - 1) / x));
}

inline int64_t workgroups_of(int64_t n_q, int G) { return ((n_q + 31) / 32 * G + 7) / 8; }

// The split that a call of these sizes may use, and the bytes its partial rows take.
inline SplitPlan plan_of(int num_seqs, int max_q, int64_t max_kv, int H_Q, int H_KV, int D, bool prompts) {
    const int64_t max_w = workgroups_of(max_q, H_Q / H_KV);
    if (max_w < 1 || max_w > 0x7fffff || fq_host::force_any_dim_attention()) return SplitPlan{0, 1};
    if (prompts && max_kv > max_q) max_kv = max_q;               // the keys beyond the queries are hidden
    return plan_split(num_seqs, H_KV, int(max_w), (max_kv + 63) / 64, fq_host::device_cu_count(), D, prompts);
}
// Workgroups that may be split, floats of their pieces' rows, and bytes of both with the number of pieces of each.
inline size_t split_slots(const SplitPlan& sp, int num_seqs, int H_KV) { return size_t(num_seqs) * H_KV * sp.split_w; }
inline size_t part_floats(const SplitPlan& sp, int num_seqs, int H_KV, int D) {
    const int slot = D == 64 ? PrefillCfg<64>::SLOT : (D == 128 ? PrefillCfg<128>::SLOT : PrefillCfg<256>::SLOT);
    return split_slots(sp, num_seqs, H_KV) * sp.max_pieces * slot;
}
inline size_t part_bytes(const SplitPlan& sp, int num_seqs, int H_KV, int D) {
    if (sp.max_pieces < 2) return 0;
    return 4 * (part_floats(sp, num_seqs, H_KV, D) + split_slots(sp, num_seqs, H_KV));
}
inline int use_plan(PrefillParams& p, const SplitPlan& sp, int D, void* workspace, size_t workspace_bytes) {
    const size_t need = part_bytes(sp, p.num_seqs, p.H_KV, D);
    p.split_w = 0;
    p.max_pieces = 1;
    p.part = nullptr;
    p.left = nullptr;
    if (need == 0 || workspace == nullptr) return FQ_OK;         // no workspace: nothing is split
    if (workspace_bytes < need) return FQ_ERR_WORKSPACE;
    if (!fq_host::aligned(workspace, 256)) return FQ_ERR_MISALIGNED;
    p.split_w = sp.split_w;
    p.max_pieces = sp.max_pieces;
    p.part = static_cast<float*>(workspace);
    p.left = reinterpret_cast<int*>(p.part + part_floats(sp, p.num_seqs, p.H_KV, D));
    return FQ_OK;
}

}  // namespace fq

extern "C" int fq_fused_tq_attention(const void* q, const uint8_t* k_packed, const float* k_norms,
                                     const uint8_t* v_packed, const float* v_norms,
                                     const float* centroids_k, const float* centroids_v,
                                     const float* rotation, int rotation_col_major, void* out,
                                     int B, int H_Q, int H_KV, int N_Q, int N_KV, int D,
                                     float sm_scale, int is_causal, int dtype, void* stream) {
    return fq_fused_tq_attention_strided(q, k_packed, k_norms, v_packed, v_norms, centroids_k, centroids_v, rotation,
                                         rotation_col_major, out, B, H_Q, H_KV, N_Q, N_KV, N_KV, N_KV, D, sm_scale,
                                         is_causal, dtype, stream);
}

extern "C" size_t fq_attention_pieces_workspace_bytes(int num_seqs, int max_q_len, int64_t max_kv_len, int H_Q, int H_KV, int D,
                                                      int prompts) {
    using namespace fq;
    if (num_seqs <= 0 || max_q_len <= 0 || max_kv_len <= 0 || H_KV <= 0 || H_Q <= 0 || H_Q % H_KV != 0) return 0;
    return part_bytes(plan_of(num_seqs, max_q_len, max_kv_len, H_Q, H_KV, D, prompts == 1 && max_q_len > 1), num_seqs, H_KV, D);
}

extern "C" size_t fq_attention_workspace_bytes(int num_seqs, int max_q_len, int64_t max_kv_len, int H_Q, int H_KV, int D,
                                               int prompts) {
    using namespace fq;
    const size_t split = fq_attention_pieces_workspace_bytes(num_seqs, max_q_len, max_kv_len, H_Q, H_KV, D, prompts);
    if (num_seqs <= 0 || max_q_len <= 0 || max_kv_len <= 0 || H_KV <= 0 || H_Q <= 0 || H_Q % H_KV != 0) return 0;
    if (prompts == 0 || !fq_host::supported_dim(D) || fq_host::force_any_dim_attention()) return split;
    const size_t expanded = plan_expanded(num_seqs, H_KV, max_q_len, max_kv_len, H_Q / H_KV, D, prompts == 1).bytes;
    return expanded > split ? expanded : split;
}

extern "C" size_t fq_paged_prefill_workspace_bytes(int num_seqs, int max_q_len, int64_t max_kv_len, int64_t total_q, int H_Q, int H_KV,
                                                   int D) {
    using namespace fq;
    const size_t split = fq_attention_pieces_workspace_bytes(num_seqs, max_q_len, max_kv_len, H_Q, H_KV, D, 0);
    if (num_seqs <= 0 || max_q_len <= 0 || max_kv_len <= 0 || H_KV <= 0 || H_Q <= 0 || H_Q % H_KV != 0) return 0;
    if (!fq_host::supported_dim(D) || fq_host::force_any_dim_attention()) return split;
    const size_t expanded = plan_expanded_paged(num_seqs, total_q, max_q_len, max_kv_len, H_KV, H_Q / H_KV, D).bytes;
    return expanded > split ? expanded : split;
}

extern "C" int fq_fused_tq_attention_strided(const void* q, const uint8_t* k_packed, const float* k_norms,
                                             const uint8_t* v_packed, const float* v_norms,
                                             const float* centroids_k, const float* centroids_v,
                                             const float* rotation, int rotation_col_major, void* out,
                                             int B, int H_Q, int H_KV, int N_Q, int N_KV,
                                             int64_t k_capacity, int64_t v_capacity, int D,
                                             float sm_scale, int is_causal, int dtype, void* stream) {
    return fq_fused_tq_attention_split(q, k_packed, k_norms, v_packed, v_norms, centroids_k, centroids_v, rotation,
                                       rotation_col_major, out, B, H_Q, H_KV, N_Q, N_KV, k_capacity, v_capacity, D, sm_scale,
                                       is_causal, dtype, nullptr, 0, stream);
}

extern "C" int fq_fused_tq_attention_split(const void* q, const uint8_t* k_packed, const float* k_norms,
                                             const uint8_t* v_packed, const float* v_norms,
                                             const float* centroids_k, const float* centroids_v,
                                             const float* rotation, int rotation_col_major, void* out,
                                             int B, int H_Q, int H_KV, int N_Q, int N_KV,
                                             int64_t k_capacity, int64_t v_capacity, int D,
                                             float sm_scale, int is_causal, int dtype, void* workspace,
                                           size_t workspace_bytes, void* stream) {
    using namespace fq;
    if (B < 0 || H_Q <= 0 || H_KV <= 0 || N_Q < 0 || N_KV < 0 || H_Q % H_KV != 0) return FQ_ERR_BAD_SHAPE;
    if (k_capacity < N_KV || v_capacity < N_KV) return FQ_ERR_BAD_SHAPE;
    if (N_KV > (1 << 24)) return FQ_ERR_BAD_SHAPE;      // the kernels address a slab's tokens with 32-bit byte offsets
    if (!fq_host::supported_dim(D)) return FQ_ERR_UNSUPPORTED_DIM;
    if (dtype != FQ_F16 && dtype != FQ_BF16) return FQ_ERR_UNSUPPORTED_DTYPE;
    if (B == 0 || N_Q == 0) return FQ_OK;
    if (N_KV == 0) return FQ_ERR_BAD_SHAPE;          // softmax over no keys is undefined
    if (!q || !k_packed || !k_norms || !v_packed || !v_norms || !centroids_k || !centroids_v || !rotation || !out)
        return FQ_ERR_NULL_POINTER;
    if (!fq_host::aligned(q, 16) || !fq_host::aligned(k_packed, 8) || !fq_host::aligned(v_packed, 4) ||
        !fq_host::aligned(rotation, 16) || !fq_host::aligned(out, 2))
        return FQ_ERR_MISALIGNED;
    if (B > 65535 || H_KV > 65535 || (D == 256 && H_Q > 65535)) return FQ_ERR_BAD_SHAPE;

    if (fq_host::force_any_dim_attention()) {
        AnyDimParams a{};
        a.q = static_cast<const uint16_t*>(q);
        a.k_packed = k_packed; a.k_norms = k_norms; a.v_packed = v_packed; a.v_norms = v_norms;
        a.centroids_k = centroids_k; a.centroids_v = centroids_v;
        a.rotation = rotation; a.rot_col_major = rotation_col_major;
        a.out = static_cast<uint16_t*>(out);
        a.H_Q = H_Q; a.H_KV = H_KV; a.G = H_Q / H_KV; a.N_Q = N_Q; a.N_KV = N_KV;
        a.k_cap = k_capacity; a.v_cap = v_capacity;
        a.causal = (is_causal && N_Q > 1) ? 1 : 0;
        a.scale_log2e = sm_scale * kLog2e;
        return launch_attention_any_dim(a, D, false, N_Q, B, dtype, stream);
    }

    const ExpandedPlan ep = plan_expanded(B, H_KV, N_Q, N_KV, H_Q / H_KV, D, is_causal && N_Q > 1);
    if (ep.per_chunk > 0 && workspace != nullptr && workspace_bytes >= ep.bytes) {
        if (!fq_host::aligned(workspace, 256)) return FQ_ERR_MISALIGNED;
        ExpandParams e{};
        e.k_packed = k_packed; e.k_norms = k_norms; e.v_packed = v_packed; e.v_norms = v_norms;
        e.centroids_k = centroids_k; e.centroids_v = centroids_v;
        e.rotation = rotation; e.rot_col_major = rotation_col_major;
        e.k_cap = k_capacity; e.v_cap = v_capacity;
        e.num_seqs = B;
        AttendParams a{};
        a.q = static_cast<const uint16_t*>(q);
        a.out = static_cast<uint16_t*>(out);
        a.H_Q = H_Q; a.H_KV = H_KV; a.G = H_Q / H_KV; a.N_Q = N_Q; a.N_KV = ep.keys;
        a.causal = (is_causal && N_Q > 1) ? 1 : 0;
        a.scale_log2e = sm_scale * kLog2e;
        a.out_wide = fq_host::aligned(out, 16);
        return launch_attention_expanded(e, a, ep, D, dtype, workspace, stream);
    }

    PrefillParams p;
    p.q = static_cast<const uint16_t*>(q);
    p.k_packed = k_packed; p.k_norms = k_norms; p.v_packed = v_packed; p.v_norms = v_norms;
    p.centroids_k = centroids_k; p.centroids_v = centroids_v;
    p.rotation = rotation; p.rot_col_major = rotation_col_major;
    p.out = static_cast<uint16_t*>(out);
    p.H_Q = H_Q; p.H_KV = H_KV; p.G = H_Q / H_KV; p.N_Q = N_Q; p.N_KV = N_KV;
    p.k_cap = k_capacity; p.v_cap = v_capacity;
    p.causal = (is_causal && N_Q > 1) ? 1 : 0;
    p.scale_log2e = sm_scale * kLog2e;

    const int64_t units = int64_t((N_Q + 31) / 32) * p.G;
    const int64_t wgs = (units + 7) / 8;
    if (wgs > 0x7fffffffLL) return FQ_ERR_BAD_SHAPE;
    const dim3 grid(static_cast<unsigned>(wgs), H_KV, B);
    hipStream_t s = static_cast<hipStream_t>(stream);
    p.cu_seqlens_q = nullptr; p.seq_lens = nullptr; p.block_table = nullptr; p.cache = nullptr;
    p.max_blocks = 0; p.num_blocks = 0; p.bs_log2 = 0;
    p.round_slots = fq_host::device_cu_count();
    p.out_wide = fq_host::aligned(out, 16);
    p.num_seqs = B;
    p.max_w = int(wgs);
    p.dense = false;
    // A launch that fills the chip keeps the plain order, one that leaves CUs idle is split if the lengths allow (here they
    // are known, and with them the pieces).
    SplitPlan sp = plan_of(B, N_Q, N_KV, H_Q, H_KV, D, p.causal != 0);
    if (sp.max_pieces > 1) {
        const SeqShape sh = make_seq_shape(N_Q, N_KV, 0, p.G, p.max_w);
        const uint32_t sum = uint32_t(B) * (uint32_t(sh.W) * uint32_t(tiles_of(sh, 0, p.G, p.causal) + tiles_of(sh, sh.W - 1, p.G, p.causal) + 1) / 2);
        const uint32_t rows = sh.W <= sp.split_w ? uint32_t(B) * uint32_t(N_Q) * uint32_t(H_Q) : 0;
        const BatchWork batch{share_of(sum * uint32_t(H_KV), p.round_slots), int(rows >> 8)};
        const int n = pieces_of(sh, batch, sp.split_w, sp.max_pieces, p.G, p.causal, D);
        sp = n < 2 ? SplitPlan{0, 1} : SplitPlan{sp.split_w, n};
    }
    const int st = use_plan(p, sp, D, workspace, workspace_bytes);
    if (st != FQ_OK) return st;
    return launch_prefill<false>(p, D, p.max_pieces > 1 ? folded_grid(int64_t(B) * H_KV * wgs * p.max_pieces) : grid, N_Q, dtype, s);
}

extern "C" int fq_paged_tq4_prefill(const void* q, const int32_t* cu_seqlens_q, const uint8_t* kv_cache,
                                    const int32_t* block_table, const int32_t* seq_lens,
                                    const float* centroids_k, const float* centroids_v,
                                    const float* rotation, int rotation_col_major, void* out,
                                    int num_seqs, int max_q_len, int H_Q, int H_KV, int D, int block_size,
                                    int max_blocks_per_seq, int64_t num_blocks, float sm_scale, int is_causal,
                                    int dtype, void* stream) {
    return fq_paged_tq4_prefill_split(q, cu_seqlens_q, kv_cache, block_table, seq_lens, centroids_k, centroids_v, rotation,
                                      rotation_col_major, out, num_seqs, max_q_len, H_Q, H_KV, D, block_size,
                                      max_blocks_per_seq, num_blocks, sm_scale, is_causal, dtype, 0, nullptr, 0, stream);
}

extern "C" int fq_paged_tq4_prefill_split(const void* q, const int32_t* cu_seqlens_q, const uint8_t* kv_cache,
                                    const int32_t* block_table, const int32_t* seq_lens,
                                    const float* centroids_k, const float* centroids_v,
                                    const float* rotation, int rotation_col_major, void* out,
                                    int num_seqs, int max_q_len, int H_Q, int H_KV, int D, int block_size,
                                    int max_blocks_per_seq, int64_t num_blocks, float sm_scale, int is_causal,
                                    int dtype, int64_t total_q, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace fq;
    if (num_seqs < 0 || max_q_len < 0 || H_Q <= 0 || H_KV <= 0 || H_Q % H_KV != 0 || max_blocks_per_seq <= 0 ||
        num_blocks <= 0 || num_blocks > 0x7fffffffLL)
        return FQ_ERR_BAD_SHAPE;
    if (!fq_host::supported_dim(D)) return FQ_ERR_UNSUPPORTED_DIM;
    if (block_size != 8 && block_size != 16 && block_size != 32) return FQ_ERR_UNSUPPORTED_BLOCK;
    if (dtype != FQ_F16 && dtype != FQ_BF16) return FQ_ERR_UNSUPPORTED_DTYPE;
    if (num_seqs == 0 || max_q_len == 0) return FQ_OK;
    if (!q || !cu_seqlens_q || !kv_cache || !block_table || !seq_lens || !centroids_k || !centroids_v || !rotation || !out)
        return FQ_ERR_NULL_POINTER;
    if (!fq_host::aligned(q, 16) || !fq_host::aligned(kv_cache, 16) || !fq_host::aligned(rotation, 16) ||
        !fq_host::aligned(out, 2))
        return FQ_ERR_MISALIGNED;
    if (num_seqs > 65535 || H_KV > 65535 || (D == 256 && H_Q > 65535)) return FQ_ERR_BAD_SHAPE;

    const ExpandedPlan ep = plan_expanded_paged(num_seqs, total_q, max_q_len, int64_t(max_blocks_per_seq) * block_size, H_KV, H_Q / H_KV, D);
    if (ep.per_chunk > 0 && workspace != nullptr && workspace_bytes >= ep.bytes && !fq_host::force_any_dim_attention()) {
        if (!fq_host::aligned(workspace, 256)) return FQ_ERR_MISALIGNED;
        ExpandParams e{};
        e.centroids_k = centroids_k; e.centroids_v = centroids_v;
        e.rotation = rotation; e.rot_col_major = rotation_col_major;
        e.cu_seqlens_q = cu_seqlens_q; e.seq_lens = seq_lens; e.block_table = block_table; e.cache = kv_cache;
        e.max_blocks = max_blocks_per_seq; e.num_blocks = int(num_blocks);
        e.bs_log2 = block_size == 8 ? 3 : (block_size == 16 ? 4 : 5);
        e.num_seqs = num_seqs;
        AttendParams a{};
        a.q = static_cast<const uint16_t*>(q);
        a.out = static_cast<uint16_t*>(out);
        a.H_Q = H_Q; a.H_KV = H_KV; a.G = H_Q / H_KV;
        a.causal = is_causal ? 1 : 0;
        a.scale_log2e = sm_scale * kLog2e;
        a.out_wide = fq_host::aligned(out, 16);
        a.paged = true;
        return launch_attention_expanded(e, a, ep, D, dtype, workspace, stream);
    }

    const int64_t wgs = workgroups_of(max_q_len, H_Q / H_KV);
    const SplitPlan sp = plan_of(num_seqs, max_q_len, int64_t(max_blocks_per_seq) * block_size, H_Q, H_KV, D, false);
    // places per KV head: every sequence of the longest kind, fewer when the tokens of the batch are known (a sequence
    // takes at most (n / 32 + 1) G / 8 + 1 workgroups), and the pieces beyond the first of those that may be split
    int64_t places = num_seqs * wgs;
    if (total_q > 0) {
        const int64_t most = (total_q / 32 + num_seqs) * (H_Q / H_KV) / 8 + num_seqs;
        places = most < places ? most : places;
    }
    // (kOrderSeqs) beyond so many sequences, and where at least half of the places of all sequences are needed, no search
    const bool dense = num_seqs > kOrderSeqs && sp.max_pieces < 2 && 2 * places >= num_seqs * wgs;
    if (dense) places = num_seqs * wgs;
    const bool fits = wgs <= 0x7fffffffLL && (places + int64_t(num_seqs) * sp.split_w * (sp.max_pieces - 1)) * H_KV <= 0x7fffffffLL;
    // (the general kernel's grid has no such bound: head_dim 256 runs there beyond it)
    if (fq_host::force_any_dim_attention() || (D == 256 && !fits)) {
        AnyDimParams a{};
        a.q = static_cast<const uint16_t*>(q);
        a.centroids_k = centroids_k; a.centroids_v = centroids_v;
        a.rotation = rotation; a.rot_col_major = rotation_col_major;
        a.out = static_cast<uint16_t*>(out);
        a.H_Q = H_Q; a.H_KV = H_KV; a.G = H_Q / H_KV;
        a.causal = is_causal ? 1 : 0;
        a.scale_log2e = sm_scale * kLog2e;
        a.cu_seqlens_q = cu_seqlens_q; a.seq_lens = seq_lens; a.block_table = block_table; a.cache = kv_cache;
        a.max_blocks = max_blocks_per_seq; a.num_blocks = int(num_blocks);
        a.bs_log2 = block_size == 8 ? 3 : (block_size == 16 ? 4 : 5);
        return launch_attention_any_dim(a, D, true, max_q_len, num_seqs, dtype, stream);
    }

    PrefillParams p;
    p.q = static_cast<const uint16_t*>(q);
    p.k_packed = nullptr; p.k_norms = nullptr; p.v_packed = nullptr; p.v_norms = nullptr;
    p.centroids_k = centroids_k; p.centroids_v = centroids_v;
    p.rotation = rotation; p.rot_col_major = rotation_col_major;
    p.out = static_cast<uint16_t*>(out);
    p.H_Q = H_Q; p.H_KV = H_KV; p.G = H_Q / H_KV; p.N_Q = 0; p.N_KV = 0;
    p.k_cap = 0; p.v_cap = 0;
    p.causal = is_causal ? 1 : 0;
    p.scale_log2e = sm_scale * kLog2e;
    p.cu_seqlens_q = cu_seqlens_q; p.seq_lens = seq_lens; p.block_table = block_table; p.cache = kv_cache;
    p.max_blocks = max_blocks_per_seq; p.num_blocks = int(num_blocks);
    p.bs_log2 = block_size == 8 ? 3 : (block_size == 16 ? 4 : 5);
    p.round_slots = fq_host::device_cu_count();
    p.out_wide = fq_host::aligned(out, 16);

    if (!fits) return FQ_ERR_BAD_SHAPE;
    p.num_seqs = num_seqs;
    p.max_w = int(wgs);
    const int st = use_plan(p, sp, D, workspace, workspace_bytes);
    if (st != FQ_OK) return st;
    p.dense = dense;
    places += int64_t(num_seqs) * p.split_w * (p.max_pieces - 1);
    return launch_prefill<true>(p, D, folded_grid(places * H_KV), max_q_len, dtype, static_cast<hipStream_t>(stream));
}
