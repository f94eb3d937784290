// Shared by the split-K paged decode kernels: the launch parameters, the chunk sizing of ragged
// long-context batches and the launch helper.
#pragma once

#include "fq_common.hpp"
#include "fq_device.hpp"

namespace fq {

struct DecodeParams {
    const void* q_rot;          // (S, H_Q, D) query dtype: rotated, or un-rotated when `rotation` is set
    int rot_col_major;          // layout of `rotation` / of the matrix given to the side kernels
    const float* rotation;      // staged kernel only: rotate the query in the prologue (NULL: already rotated)
    const float* sketch;        // TurboQuantProd pages only: the (D, D) sign-sketch matrix S
    const uint8_t* cache;       // (num_blocks, BS, H_KV*(D+8))
    const int32_t* block_table; // (S, max_blocks)
    const int32_t* seq_lens;    // (S,)
    const float* centroids_k;
    const float* centroids_v;
    float* part_acc;            // (S, H_Q, NS, D)
    float* part_m;              // (S, H_Q, NS)
    float* part_l;              // (S, H_Q, NS)
    int H_Q, H_KV, G;           // G = H_Q / H_KV
    int max_blocks;
    int num_blocks;
    int num_splits;
    int two_tables;             // centroids_v differs from centroids_k
    float scale_log2e;          // sm_scale * log2(e)
    int heads_per_wg;           // direct kernel: KV heads a workgroup serves; its other wavefronts take further splits
    int spin_limit;             // staged kernel: polls of a bounded wait between wavefronts before it gives up
    int balance_slots;          // staged kernel: > 0 lets the workgroups size the token chunks from the actual
                                // sequence lengths, for this many workgroups running at a time (num_seqs <= kBalanceSeqs)
    // Staged kernel instantiated with STORE: the serving step in one launch.  The workgroup whose split
    // holds a sequence's last token first compresses that token's new key and value rows into their
    // cache row (slot new_slots[seq]; negative: not stored), then reads the row back with its tile.
    uint8_t* cache_rw;          // the cache again, for the row that is written
    const void* new_key;        // (S, H_KV, D) query dtype, one token per sequence
    const void* new_value;
    const int64_t* new_slots;   // (S,) flat slot of the new token
    const float* boundaries;    // (15,) ascending
    int64_t num_slots;          // num_blocks * block_size
};


// Sum of the lanes up to and including this one.
__device__ __forceinline__ int wave_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);    // row_shr:1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);    // row_bcast:15 to rows 1 and 3, :31 to rows 2 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
    return v;
}

// x / d rounded up, both below 2^24 and the quotient below 2^18, rc about 1 / d (a division of integers takes four times the
// instructions).
__device__ __forceinline__ int quotient_up(int x, int d, float rc) {
    const int q = int(float(x) * rc), r = x - q * d;           // q is off by one at most
    return q + (r > 0 ? 1 : 0) + (r > d ? 1 : 0) - (r <= -d ? 1 : 0);
}

// balance_chunks for 65 to 256 sequences, four a lane: nine candidates (lane j holds the j-th; eight in steps of an eighth of the
// smallest chunk, rounded up to 64 rows, and exactly twice the smallest), the workgroups of two of them added up at a time.
// The cost of a candidate is that of its rounds of workgroups as long as the longest, or, where most are shorter, of a CU's share
// of all rows and prologues and the longest workgroup on top (256 sequences of which one has 2048 tokens and the others at most
// 340: 59 us, and 96 with the rounds alone, which saw 257 workgroups of 1024 rows against 256 of 2048).
// Every workgroup pays for this, also one without work and one of a batch that nothing helps, so it is short: where the
// smallest chunk makes one round, or is the best and leaves no pair without work, all stays as it was.  Twice the smallest
// chunk is what a batch of equal lengths in an even number of rounds gains by, half the rounds with a prologue less.
template <int TPR>
__device__ __forceinline__ void balance_chunks_many(const DecodeParams& p, int lane, int NS, int cap, int max_tokens, int& chunk,
                                                    int& seq, int& split, int& L_known) {
    constexpr int K = 4, CANDS = 9;
    const int nseq = int(gridDim.x);
    int l_real[K], rows[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int at = K * lane + k;
        const int l = p.seq_lens[at < nseq ? at : nseq - 1];
        l_real[k] = at >= nseq || l < 0 ? 0 : (l > max_tokens ? max_tokens : l);
        rows[k] = (l_real[k] + TPR - 1) / TPR;
    }
    int cand = lane >= CANDS - 1 ? 2 * chunk : chunk + lane * (((chunk >> 3) + 63) & ~63);
    cand = cand < cap ? cand : cap;
    cand = cand > chunk ? cand : chunk;
    const int rc_mine = int(__builtin_bit_cast(uint32_t, __builtin_amdgcn_rcpf(float(cand))));
    auto rc_of = [&](int j) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(rc_mine, j)); };
    auto groups_of = [&](int j) {                              // (the host sees to it that 16 bits hold the sum)
        const float rc = rc_of(j);
        float n = 0.0f;
#pragma unroll
        for (int k = 0; k < K; ++k) n += __builtin_ceilf(float(rows[k]) * rc - 0.0009765625f);
        return uint32_t(n);
    };
    auto length_of = [&](int sq) {
        int l = 0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int lk = __builtin_amdgcn_readlane(l_real[k], sq / K);
            l = sq % K == k ? lk : l;
        }
        return l;
    };
    const uint32_t smallest = wave_sum(groups_of(0));
    int best = 0;
    if (int(smallest) > p.balance_slots) {
        uint32_t mine = smallest, total = 0;
        float longest = 0.0f;
#pragma unroll
        for (int j = 1; j < CANDS; j += 2) {
            const uint32_t both = wave_sum(groups_of(j) | groups_of(j + 1) << 16);
            mine = lane == j ? both & 0xffffu : (lane == j + 1 ? both >> 16 : mine);
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
            total += uint32_t(rows[k]);
            longest = __builtin_fmaxf(longest, float(rows[k]));
        }
        const float per_slot = __builtin_amdgcn_rcpf(float(p.balance_slots)), n = float(mine);
        const float work = (float(wave_sum(total)) + 96.0f * n) * per_slot;
        const float rounds = __builtin_ceilf(n * per_slot - 0.0009765625f);
        const float largest = __builtin_fminf(float(cand), wave_max(longest)) + 96.0f;
        const float cost = lane < CANDS ? __builtin_fminf(__builtin_fmaxf(rounds, 1.0f) * largest, work + largest) : __builtin_inff();
        const uint64_t cheapest = __ballot(cost == -wave_max(-cost));
        best = __ffsll(static_cast<unsigned long long>(cheapest)) - 1;
    }
    if (int(smallest) <= p.balance_slots || (best == 0 && int(smallest) == nseq * NS)) {
        L_known = length_of(seq);
        return;
    }
    chunk = __builtin_amdgcn_readlane(cand, best);
    const float rc = rc_of(best);
    int n[K], live = 0, dead = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        n[k] = quotient_up(rows[k], chunk, rc);
        n[k] = n[k] < NS ? n[k] : NS;
        live += n[k];
        dead += K * lane + k < nseq ? NS - n[k] : 0;
    }
    // the w-th of the live pairs, else of the empty ones: the lane that holds it, then which of its sequences
    const int live_incl = wave_scan(live);
    const int total_live = __builtin_amdgcn_readlane(live_incl, 63);
    const int w = int(blockIdx.x) + int(gridDim.x) * int(blockIdx.y);
    const bool is_live = w < total_live;
    const int incl = is_live ? live_incl : wave_scan(dead), e = is_live ? w : w - total_live;
    int sl = __builtin_popcountll(__ballot(incl <= e));
    sl = sl < (nseq - 1) / K ? sl : (nseq - 1) / K;
    int rem = e - __builtin_amdgcn_readlane(incl - (is_live ? live : dead), sl);
    seq = -1;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int nk = __builtin_amdgcn_readlane(n[k], sl), have = is_live ? nk : NS - nk;
        const bool last = K * sl + k >= nseq - 1 || k == K - 1;
        if (seq < 0 && (rem < have || last)) {
            seq = K * sl + k;
            split = is_live ? rem : nk + rem;
        }
        rem -= have;
    }
    split = split < NS ? split : NS - 1;
    L_known = length_of(seq);
}

// Most sequences of a batch whose chunks follow from the actual lengths.
constexpr int kBalanceSeqs = 256;

// Ragged batches of long contexts (at most 64 sequences here, one lane each; more above).  With the chunk
// of the longest possible context the live workgroups are all the same size and their
// count is whatever the lengths add up to, e.g. 2.1 rounds over the chip, which costs 3.
// Every workgroup evaluates the same 64 candidate chunk sizes (one per lane) on the
// actual lengths, cost = rounds x (chunk + a prologue's worth of tokens), and takes the
// cheapest: same inputs, same arithmetic, same answer in every workgroup.  Larger chunks
// only: the split count bounds the chunk from below.  On return `chunk` is the chosen size,
// (`seq`, `split`) the pair this workgroup takes and `L_known` its sequence's length.
// TPR: tokens per row of the kernel (rows of 2, 4 or 8 consecutive tokens when the model has 4, 2 or 1 KV heads)
template <int PVR, int BS, int TPR>
__device__ __forceinline__ void balance_chunks(const DecodeParams& p, int lane, int NS, bool rowwide, int& chunk, int& seq,
                                               int& split, int& L_known) {
    const int cap = rowwide ? chunk * NS : 64 * PVR * BS;       // page ids of a split: 64 * PVR lanes
    if (int(gridDim.x) > kWave)
        return balance_chunks_many<TPR>(p, lane, NS, cap, p.max_blocks * BS * TPR, chunk, seq, split, L_known);
    const int step = ((chunk >> 4) + 63) & ~63;
    int cand = chunk + lane * step;
    cand = cand < cap ? cand : cap;
    cand = cand > chunk ? cand : chunk;
    const float rc = __builtin_amdgcn_rcpf(float(cand));
    const int nseq = int(gridDim.x);
    int l_real = lane < nseq ? p.seq_lens[lane] : 0;
    l_real = l_real < 0 ? 0 : (l_real > p.max_blocks * BS * TPR ? p.max_blocks * BS * TPR : l_real);
    const int l_mine = (l_real + TPR - 1) / TPR;               // in rows
    float groups = 0.0f;
    for (int sq = 0; sq < nseq; ++sq)
        groups += __builtin_ceilf(float(__builtin_amdgcn_readlane(l_mine, sq)) * rc - 0.0009765625f);
    const float rounds = __builtin_ceilf(groups * __builtin_amdgcn_rcpf(float(p.balance_slots)) - 0.0009765625f);
    const float cost = (rounds < 1.0f ? 1.0f : rounds) * float(cand + 96);
    uint32_t key = (uint32_t(cost) << 6) | uint32_t(lane);
#pragma unroll
    for (int mask = 1; mask < 64; mask <<= 1) {
        const uint32_t other = uint32_t(__shfl_xor(int(key), mask, kWave));
        key = other < key ? other : key;
    }
    const int best = chunk + int(key & 63u) * step;
    chunk = best < cap ? best : (cap > chunk ? cap : chunk);

    // The live (sequence, split) pairs first, in sequence order, then the empty ones: the w-th
    // workgroup of the grid takes the w-th pair of that list.  Live workgroups are all of one
    // size and now consecutive, so they spread evenly over the XCDs and CUs whatever the lengths.
    auto scan = [&](int v) {
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int t = __shfl_up(v, d, kWave);
            v += lane >= d ? t : 0;
        }
        return v;
    };
    int n_mine = lane < nseq ? (l_mine + chunk - 1) / chunk : 0;
    n_mine = n_mine < NS ? n_mine : NS;
    const int live_incl = scan(n_mine);
    const int total_live = __builtin_amdgcn_readlane(live_incl, 63);
    const int w = int(blockIdx.x) + int(gridDim.x) * int(blockIdx.y);
    if (w < total_live) {
        const int s_idx = __builtin_popcountll(__ballot(live_incl <= w));
        seq = s_idx;
        split = w - __builtin_amdgcn_readlane(live_incl - n_mine, s_idx);
    } else {
        const int e = w - total_live;
        const int dead_mine = lane < nseq ? NS - n_mine : 0;
        const int dead_incl = scan(dead_mine);
        int s_idx = __builtin_popcountll(__ballot(dead_incl <= e));
        s_idx = s_idx < nseq ? s_idx : nseq - 1;
        seq = s_idx;
        split = __builtin_amdgcn_readlane(n_mine, s_idx) + (e - __builtin_amdgcn_readlane(dead_incl - dead_mine, s_idx));
        split = split < NS ? split : NS - 1;
    }
    L_known = __builtin_amdgcn_readlane(l_real, seq);
}

// Launch with `lds` bytes of dynamic LDS; more than 64 KB per workgroup has to be
// allowed per kernel function first.
template <typename K>
inline int launch_with_lds(K kernel, const DecodeParams& p, dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
    if (lds > 32768 && !fq_host::lds_limit_raised(reinterpret_cast<const void*>(kernel), lds)) return FQ_ERR_LAUNCH;
    hipLaunchKernelGGL(kernel, grid, block, lds, stream, p);
    return fq_host::check_launch();
}

// The ring kernel (fq_paged_decode_ring.hip): groups of 8 KV heads of dimension 128, TQ4 pages.
int launch_ring(const DecodeParams& p, int num_seqs, int block_size, bool wide, int dtype, hipStream_t stream);

}  // namespace fq
