// Attention of many queries over packed TQ4 keys and values (fused_tq_attention_reference,
// src/flashquant/kernels/cpu_reference.py:154-227), in two launches.  Where several workgroups read the same keys, what the
// kernel of fq_fused_attention.hip does for every one of them is done once:
//   tq4_expand_kernel       keys and values rotated back to the original space, as fp16 in the order in which the products
//                           below read them:   image = (centroid[idx] @ R) * norm
//   attend_expanded_kernel  plain attention over these: no tables, no rotation of the query or of the output
// since (q R^T) . k = q . (k R) and (sum w v) R = sum w (v R).  The query is not rounded once more on the way, and a key or value
// is rounded as its centroids and once at the end (there: centroids, norm and product): error against 64 bits, causal,
// 1000 x 8 heads over 2 of 128 coordinates, fp16 7.7e-4 there and 5.0e-4 here, bf16 2.6e-3 and 1.7e-3.
#include "fq_attention_expanded.hpp"

#include <type_traits>

#include "fq_common.hpp"
#include "fq_device.hpp"

namespace fq {

namespace {

// The image of a tile: 1 KB blocks, one 16-byte operand of v_mfma_f32_32x32x16_f16 a lane, so that LDS takes them as they lie and
// reads them without conflicts and with one address.  Keys: block (32 tokens, 16 coordinates); values: (16 tokens, 32 coordinates),
// the tokens in the order in which the scores of a lane lie in its registers.
template <int D>
struct TileCfg {
    static constexpr int TS = D == 256 ? 5 : 6;
    static constexpr int TT = 1 << TS;
    static constexpr int NKS = D / 16;
    static constexpr int NOB = D / 32;
    static constexpr int NTB = TT / 32, NVS = TT / 16;
    static constexpr int SIDE = TT * D * 2;
    static constexpr int TILE = 2 * SIDE;
    static constexpr int ROUNDS = D == 256 ? 4 : 1;
    static constexpr int RB = NOB / ROUNDS;
    static constexpr int RTERM = NKS * RB * 1024;
    static constexpr int UNIT = 32 * D + 64;               // floats of a unit's piece: its rows, 32 maxima, 32 sums
};

// Coordinate (of 32) in row r of a matrix operand: result register e of lane half h is then coordinate 16 (e / 8) + 8 h + e % 8.
__device__ __forceinline__ int coord_of_row(int r) { return 16 * (r >> 4) + 8 * ((r >> 2) & 1) + 4 * ((r >> 3) & 1) + (r & 3); }

typedef uint4v uint4a __attribute__((aligned(4)));

// Rows of a norm n are at most n * span * sqrt(D) long (`span`: the largest centroid).  Those of 2^14 and more are stored divided
// by a power of two, which leaves room for a matrix whose columns are up to 4 long.
template <int D>
__device__ __forceinline__ int reach_of(float span) {
    const float len = span * (D == 64 ? 8.0f : (D == 128 ? 11.4f : 16.0f));
    return int((float_to_bits(len) >> 23) & 0xffu) - 126;
}
__device__ __forceinline__ int row_excess(float n, int reach) {
    const int ex = int((float_to_bits(n) >> 23) & 0xffu) - 126 + reach;
    return ex > 14 ? ex - 14 : 0;
}

// A sequence as the launches see it.
struct Seq {
    int NQ, NKV, q_first, qoff;
    __device__ __forceinline__ int tiles(int ts) const { return NQ > 0 ? (NKV + (1 << ts) - 1) >> ts : 0; }
};
template <bool PAGED>
__device__ __forceinline__ Seq seq_of(const ExpandParams& p, int s) {
    if (!PAGED) return Seq{p.N_Q, p.keys, 0, 0};
    const int first = p.cu_seqlens_q[s], nq = p.cu_seqlens_q[s + 1] - first, room = p.max_blocks << p.bs_log2;
    int nkv = p.seq_lens[s];
    nkv = nkv < 0 ? 0 : (nkv > room ? room : nkv);
    return Seq{nq > 0 ? nq : 0, nkv, first, nkv > nq ? nkv - nq : 0};
}

// Sum over the lanes up to this one.
__device__ __forceinline__ int wave_scan(int v, int lane) {
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int u = __shfl_up(v, d, kWave);
        if (lane >= d) v += u;
    }
    return v;
}

// The work of the second launch, by one workgroup while the others expand: the workgroups of all sequences (128 rows each), those
// of more tiles than a CU's share in pieces of at most that, in classes of a third of a binary order of their length, the longest
// first, and in a class in the order of the sequences (their keys then stay in the L2).
constexpr int kPlanClasses = 16;
template <int D, bool PAGED>
__device__ void make_plan(const ExpandParams& p, int* lds) {
    constexpr int TS = TileCfg<D>::TS;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int* wfirst = lds;                          // first workgroup of a sequence, [num_seqs]: all
    int* tfirst = lds + 260;                    // first tile
    int* sums = lds + 520;                      // of the wavefronts
    int64_t* parts = reinterpret_cast<int64_t*>(lds + 560);
    int* hist = lds + 640;                      // pieces by (class, thread)
    auto block_scan = [&](int v, int& total) {  // sum over the threads up to this one, and over all
        const int incl = wave_scan(v, lane);
        __syncthreads();
        if (lane == 63) sums[wave] = incl;
        __syncthreads();
        int before = 0;
        total = 0;
        for (int i = 0; i < 8; ++i) {
            before += i < wave ? sums[i] : 0;
            total += sums[i];
        }
        return before + incl;
    };
    auto block_sum = [&](int64_t v) {
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) v += __shfl_xor(v, d, kWave);
        __syncthreads();
        if (lane == 0) parts[wave] = v;
        __syncthreads();
        int64_t total = 0;
        for (int i = 0; i < 8; ++i) total += parts[i];
        return total;
    };
    auto tiles_of = [&](const Seq& q, int x) {  // that the workgroup's last row sees
        const int all = (q.NKV + (1 << TS) - 1) >> TS, units = ((q.NQ + 31) >> 5) * p.G;
        if (!p.causal) return all;
        const int last = 4 * x + 3 < units - 1 ? 4 * x + 3 : units - 1;
        int pos = 32 * (last / p.G) + 31;
        pos = pos < q.NQ - 1 ? pos : q.NQ - 1;
        const int t = ((q.qoff + pos) >> TS) + 1;
        return t < all ? t : all;
    };
    int W = 0, tiles = 0, most = 0;
    int64_t work = 0;
    if (tid < p.num_seqs) {
        const Seq q = seq_of<PAGED>(p, tid);
        W = (((q.NQ + 31) >> 5) * p.G + 3) >> 2;
        tiles = q.tiles(TS);
        most = W > 0 ? tiles_of(q, W - 1) : 0;
        work = W > 0 ? work_of(W, tiles_of(q, 0), most) : 0;
    }
    int groups, all_tiles;
    const int wincl = block_scan(W, groups), tincl = block_scan(tiles, all_tiles);
    const int64_t all_work = block_sum(work);
    if (tid < p.num_seqs) {
        wfirst[tid] = wincl - W;
        tfirst[tid] = tincl - tiles;
    }
    __syncthreads();
    if (lane == 0) sums[wave] = 0;
    const int longest_here = int(wave_max(float(most)));
    __syncthreads();
    if (lane == 0) sums[wave] = longest_here;
    __syncthreads();
    int longest = 1;
    for (int i = 0; i < 8; ++i) longest = longest > sums[i] ? longest : sums[i];
    const int per = (groups + 511) / 512;
    auto each = [&](auto&& f) {                 // this thread's workgroups, in order
        int s = 0;
        for (int i = tid * per; i < (tid + 1) * per && i < groups; ++i) {
            int lo = s, hi = p.num_seqs;        // wfirst[lo] <= i < wfirst[hi]
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (wfirst[mid] <= i) lo = mid;
                else hi = mid;
            }
            s = lo;
            const Seq q = seq_of<PAGED>(p, s);
            const int end = s + 1 < p.num_seqs ? wfirst[s + 1] : groups;
            f(s, q, end - 1 - i, tiles_of(q, end - 1 - i));
        }
    };
    const int64_t share = share_of_work(all_work, p.H_KV, p.plan.cu_slots);
    auto pieces_of = [&](int t, int piece) { return t <= piece ? 1 : (t + piece - 1) / piece; };
    int piece = longest;
    int64_t best = 0;
    for (int i = 0; i < kPieceChoices && (i == 0 || p.plan.max_slots > 0); ++i) {
        const int choice = piece_choice(i, longest, kPieceTiles << (6 - TS));
        int n = 0, n_split = 0, all, all_split;
        each([&](int, const Seq&, int, int t) {
            const int k = pieces_of(t, choice);
            n += k;
            n_split += k > 1 ? k : 0;
        });
        block_scan(n, all);
        block_scan(n_split, all_split);
        if (i > 0 && (all > p.plan.max_items || all_split > p.plan.max_slots)) break;
        const int64_t ns = batch_ns(choice, share, int64_t(all) * p.H_KV, int64_t(all_split) * p.H_KV, p.plan.cus, D, !PAGED && !p.causal);
        if (i == 0 || 20 * ns < 19 * best) {
            best = ns;
            piece = choice;
        }
        if (choice <= (kPieceTiles << (6 - TS))) break;
    }
    auto class_of = [&](int len) {              // 0: the longest pieces
        const float r = 3.0f * __log2f(float(piece < longest ? piece : longest) / float(len > 0 ? len : 1));
        const int c = int(r);
        return c < 0 ? 0 : (c < kPlanClasses ? c : kPlanClasses - 1);
    };
    for (int c = 0; c < kPlanClasses; ++c) hist[c * 512 + tid] = 0;
    int slots = 0, split = 0;
    each([&](int, const Seq&, int, int t) {
        const int k = pieces_of(t, piece);
        hist[class_of((t + k - 1) / k) * 512 + tid] += k;
        slots += k > 1 ? k : 0;
        split += k > 1 ? 1 : 0;
    });
    int all, all_slots, all_split;
    const int slot_incl = block_scan(slots, all_slots), split_incl = block_scan(split, all_split);
    __syncthreads();
    int here[kPlanClasses], mine = 0;           // 16 neighbours of the table a thread
    for (int c = 0; c < kPlanClasses; ++c) {
        here[c] = hist[tid * kPlanClasses + c];
        mine += here[c];
    }
    int at = block_scan(mine, all) - mine;
    for (int c = 0; c < kPlanClasses; ++c) {
        hist[tid * kPlanClasses + c] = at;
        at += here[c];
    }
    __syncthreads();
    int slot = slot_incl - slots, split_at = split_incl - split;
    each([&](int s, const Seq& q, int x, int t) {
        const int k = pieces_of(t, piece);
        WorkPiece w{s, q.q_first, q.NQ, q.NKV, x, k, PAGED ? tfirst[s] : 0, slot};
        int& to = hist[class_of((t + k - 1) / k) * 512 + tid];
        if (k > 1) p.plan.splits[split_at++] = w;
        for (int i = 0; i < k; ++i, ++to) {
            w.x = x | i << 20;
            if (to < p.plan.max_items) p.plan.items[to] = w;    // (more only where cu_seqlens_q goes beyond the tokens)
        }
        slot += k > 1 ? k : 0;
    });
    if (tid == 0) {
        p.plan.counts[0] = all < p.plan.max_items ? all : p.plan.max_items;
        p.plan.counts[1] = all_split;
    }
}

// An item is TBI blocks of 32 tokens of the keys or the values of a pair, on one wavefront from the packed rows to the image, with no
// barrier: lookups (pair table as in the other kernels) into matrix operands, the products with both terms of the matrix out of
// LDS (two fp16 terms of 256 R: 2^-22 of its largest entry), the norm in float32, one rounding.  A lane's half row is contiguous
// (the contraction index is permuted on both sides), its result registers are whole operands of the image.  At 256 coordinates
// the matrix is 256 KB and blockIdx.y has a quarter of the columns.
// Bound by the stores where there are many tiles (4 x 8 heads x 8192 tokens of 128 45 us, 134 MB), by the start (5.3 us: matrix
// and tables) and one item's chain where there are few: 8 heads x 65 tokens 7.6 us.  Stores that stay out of the L2 (nontemporal)
// 18.9 -> 15.6 us at 128 pairs x 300 tokens: else they are written back at the end of the launch.
template <int D, int TBI, bool PAGED, bool PLANNED>
__global__ __launch_bounds__(512) void tq4_expand_kernel(const ExpandParams p) {
    using C = TileCfg<D>;
    constexpr int NKS = C::NKS, NTB = TBI, RB = C::RB, TT = C::TT, HT = TT / 32, IPT = HT / TBI, BPW = RB * NKS / 8;
    constexpr int DW = NKS;                                  // packed dwords of a lane's half row
    extern __shared__ __attribute__((aligned(256))) uint8_t lds[];
    uint32_t* lut = reinterpret_cast<uint32_t*>(lds);
    uint8_t* rot = lds + 65536;
    const int tid = threadIdx.x, lane = tid & 63, m32 = lane & 31, hf = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int round = blockIdx.y;
    const int stride = int(gridDim.x) - (PLANNED ? 1 : 0);
    if constexpr (PLANNED) {
        if (int(blockIdx.x) == stride) {
            if (round == 0) make_plan<D, PAGED>(p, reinterpret_cast<int*>(lds));
            return;
        }
    }
    // the first tiles of the sequences 64 i + lane
    int firsts[PAGED ? 4 : 1];
    int tiles = p.pairs * p.tiles;
    if constexpr (PAGED) {
        tiles = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int mine = 64 * i + lane < p.num_seqs ? seq_of<PAGED>(p, 64 * i + lane).tiles(C::TS) : 0;
            const int incl = wave_scan(mine, lane);
            firsts[i] = tiles + incl - mine;
            tiles += __builtin_amdgcn_readlane(incl, 63);
        }
        tiles *= p.H_KV;
    }
    const int items = tiles * 2 * IPT;

    uint4v raw[NTB][DW / 4];
    float nrm[NTB];
    auto issue = [&](int item_raw) {
        const int item = item_raw < items ? item_raw : items - 1;
        const int side = item & 1, part = (item >> 1) % IPT, at = (item >> 1) / IPT;
        if constexpr (PAGED) {
            const int g = at / p.H_KV, hkv = at - g * p.H_KV;
            int s = -1;                                      // the last sequence whose first tile is not behind this one
#pragma unroll
            for (int i = 0; i < 4; ++i) s += __popcll(__ballot(64 * i + lane < p.num_seqs && firsts[i] <= g));
            int first = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if ((s >> 6) == i) first = __builtin_amdgcn_readlane(firsts[i], s & 63);
            const int keys = seq_of<PAGED>(p, s).NKV;
            const int64_t row_bytes = int64_t(p.H_KV) * (D + 8);
#pragma unroll
            for (int tb = 0; tb < NTB; ++tb) {
                const int t_raw = (g - first) * TT + 32 * (TBI * part + tb) + m32, t = t_raw < keys ? t_raw : keys - 1;
                int pg = p.block_table[int64_t(s) * p.max_blocks + (t >> p.bs_log2)];
                pg = pg < 0 ? 0 : (pg >= p.num_blocks ? p.num_blocks - 1 : pg);
                const uint8_t* row = p.cache + ((int64_t(pg) << p.bs_log2) + (t & ((1 << p.bs_log2) - 1))) * row_bytes + side * p.H_KV * (D / 2 + 4);
#pragma unroll
                for (int i = 0; i < DW / 4; ++i) raw[tb][i] = *reinterpret_cast<const uint4a*>(row + hkv * (D / 2) + hf * (D / 4) + 16 * i);
                nrm[tb] = *reinterpret_cast<const float*>(row + p.H_KV * (D / 2) + 4 * hkv);
                if (t_raw >= keys) nrm[tb] = 0.0f;
            }
            return;
        }
        const int tile = at % p.tiles, pair = p.pair0 + at / p.tiles;
        const uint8_t* packed = side ? p.v_packed + int64_t(pair) * p.v_cap * (D / 2) : p.k_packed + int64_t(pair) * p.k_cap * (D / 2);
        const float* norms = side ? p.v_norms + int64_t(pair) * p.v_cap : p.k_norms + int64_t(pair) * p.k_cap;
#pragma unroll
        for (int tb = 0; tb < NTB; ++tb) {
            const int t_raw = tile * TT + 32 * (TBI * part + tb) + m32, t = t_raw < p.keys ? t_raw : p.keys - 1;
            const uint8_t* row = packed + (uint32_t(t) * uint32_t(D / 2) + uint32_t(hf) * (D / 4));
#pragma unroll
            for (int i = 0; i < DW / 4; ++i) raw[tb][i] = *reinterpret_cast<const uint4a*>(row + 16 * i);
            nrm[tb] = norms[t];
            if (t_raw >= p.keys) nrm[tb] = 0.0f;
        }
    };

    const float cent_k = p.centroids_k[lane & 15], cent_v = p.centroids_v[lane & 15];
    float rbv[BPW][8];
#pragma unroll
    for (int i = 0; i < BPW; ++i) {
        const int blk = BPW * w + i, j = 32 * (RB * round + blk / NKS) + coord_of_row(m32), k0 = hf * (D / 2) + 8 * (blk % NKS);
        if (p.rot_col_major) {
            const float4v lo = *reinterpret_cast<const float4v*>(p.rotation + j * D + k0);
            const float4v hi = *reinterpret_cast<const float4v*>(p.rotation + j * D + k0 + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) { rbv[i][e] = lo[e]; rbv[i][4 + e] = hi[e]; }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) rbv[i][e] = p.rotation[(k0 + e) * D + j];
        }
    }
    int item = int(blockIdx.x) + stride * w;
    if (items > 0) issue(item);
    fill_pair_tables<8>(lut, cent_k, cent_v, 15, w, lane);
#pragma unroll
    for (int i = 0; i < BPW; ++i) {
        half8 hi, lo;
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const float a = rbv[i][e] * 256.0f, b = rbv[i][e + 1] * 256.0f;
            const auto h2 = __builtin_amdgcn_cvt_pkrtz(a, b);
            const auto l2 = __builtin_amdgcn_cvt_pkrtz(a - float(h2[0]), b - float(h2[1]));
            hi[e] = h2[0]; hi[e + 1] = h2[1];
            lo[e] = l2[0]; lo[e + 1] = l2[1];
        }
        *reinterpret_cast<half8*>(rot + ((BPW * w + i) * 64 + lane) * 16) = hi;
        *reinterpret_cast<half8*>(rot + C::RTERM + ((BPW * w + i) * 64 + lane) * 16) = lo;
    }
    const float span_k = wave_max(__builtin_fabsf(cent_k)), span_v = wave_max(__builtin_fabsf(cent_v));
    const int reach_k = reach_of<D>(span_k), reach_v = reach_of<D>(span_v);
    __syncthreads();

    const uint8_t* rsrc = rot + 16 * lane;
    for (; item < items; item += 8 * stride) {
        const int side = item & 1, part = (item >> 1) % IPT, at = (item >> 1) / IPT;     // (pair, tile) of this launch
        const uint32_t lane_off = 4u * uint32_t(m32) + 128u * uint32_t(side);
        half8 tok[NTB][NKS];
        float scale[NTB];
        int over[NTB];
#pragma unroll
        for (int tb = 0; tb < NTB; ++tb) {
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) tok[tb][ks] = __builtin_bit_cast(half8, lookup_word(lds, raw[tb][ks >> 2][ks & 3], lane_off));
            over[tb] = row_excess(nrm[tb], side ? reach_v : reach_k);
            const float n = __builtin_ldexpf(nrm[tb], -over[tb] - 8);
            scale[tb] = __builtin_fabsf(n) < __builtin_inff() ? n : __builtin_nanf("");
        }
        // (`flags` and `exps`: by pair, tile, side and block of 32 tokens)
        if (round == 0) {
#pragma unroll
            for (int tb = 0; tb < NTB; ++tb) {
                const int64_t block = (int64_t(at) * 2 + side) * HT + TBI * part + tb;
                const bool big = __any(over[tb] != 0);
                if (lane == 0) p.flags[block] = big ? 1 : 0;
                if (big && hf == 0) p.exps[block * 32 + m32] = over[tb];
            }
        }
        issue(item + 8 * stride);
        float vs[NTB][16];                                   // of the tokens in a lane's result registers (values)
        if (side) {
#pragma unroll
            for (int tb = 0; tb < NTB; ++tb)
#pragma unroll
                for (int r = 0; r < 16; ++r) vs[tb][r] = __shfl(scale[tb], 8 * (r >> 2) + 4 * hf + (r & 3), kWave);
        }
        uint8_t* img = p.images + int64_t(at) * C::TILE + side * C::SIDE + 16 * lane;
#pragma unroll
        for (int cb = 0; cb < RB; ++cb) {
            float16v acc[NTB] = {};
            if (side) {
#pragma unroll
                for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
                    for (int term = 0; term < 2; ++term) {
                        const half8 r = *reinterpret_cast<const half8*>(rsrc + term * C::RTERM + (cb * NKS + ks) * 1024);
#pragma unroll
                        for (int tb = 0; tb < NTB; ++tb) acc[tb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(tok[tb][ks], r, acc[tb], 0, 0, 0);
                    }
            } else {
#pragma unroll
                for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
                    for (int term = 0; term < 2; ++term) {
                        const half8 r = *reinterpret_cast<const half8*>(rsrc + term * C::RTERM + (cb * NKS + ks) * 1024);
#pragma unroll
                        for (int tb = 0; tb < NTB; ++tb) acc[tb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(r, tok[tb][ks], acc[tb], 0, 0, 0);
                    }
            }
            const int ob = RB * round + cb;
#pragma unroll
            for (int tb = 0; tb < NTB; ++tb)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    uint4v o;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int r = 8 * u + 2 * e;
                        const float s0 = side ? vs[tb][r] : scale[tb], s1 = side ? vs[tb][r + 1] : scale[tb];
                        o[e] = round_pair<FQ_F16>(acc[tb][r] * s0, acc[tb][r + 1] * s1);
                    }
                    const int block = TBI * part + tb, blk = side ? (2 * block + u) * C::NOB + ob : block * NKS + 2 * ob + u;
                    __builtin_nontemporal_store(o, reinterpret_cast<uint4v*>(img + blk * 1024));
                }
        }
    }
}

// Two workgroups a CU, so that one computes where the other waits; at 256 coordinates a wavefront takes 380 registers.
template <int D>
struct AttendCfg {
    static constexpr int WAVES = D == 256 ? 1 : 2, NBUF = D == 256 ? 4 : 2;
};

// What a wavefront has to do: 32 positions of one query head, over some of the tiles they see.  Positions, keys and tiles count
// from the first of these tiles.
struct Rows {
    int64_t q0;                         // element of the first position's row, and
    int q_stride;                       // from one position to the next
    int at, step;                       // image of the first tile; images from one tile to the next
    int row0, NQ, pos0, NKV, w;         // first row and rows of the sequence; position of the first row, keys
    int ntiles, my_tiles, full;         // of the workgroup; of this wavefront; that hide nothing from its rows
    int pieces, slot;                   // of the workgroup; where the rows of this piece go
    bool live, none;
};

template <int D, bool PLANNED>
__device__ __forceinline__ Rows rows_of(const AttendParams& p) {
    using C = TileCfg<D>;
    constexpr int TT = C::TT, TS = C::TS;
    Rows r{};
    const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    r.w = w;
    int b, hkv, x, qoff = 0, piece = 0, q_first = 0, NKV = p.N_KV;
    r.NQ = p.N_Q;
    r.pieces = 1;
    const bool paged = PLANNED && p.paged;
    if constexpr (PLANNED) {
        const int place = int(blockIdx.x) / p.H_KV;
        hkv = int(blockIdx.x) % p.H_KV;
        r.none = place >= p.plan.counts[0];
        if (r.none) return r;
        const WorkPiece wp = p.plan.items[place];
        b = wp.seq; x = wp.x & 0xfffff; piece = wp.x >> 20;
        r.NQ = wp.NQ; NKV = wp.NKV; r.pieces = wp.pieces; q_first = wp.q_first;
        r.slot = (wp.slot + piece) * p.H_KV + hkv;
        qoff = paged && NKV > r.NQ ? NKV - r.NQ : 0;
        r.at = paged ? wp.tile_base * p.H_KV + hkv : (b * p.H_KV + hkv) * p.tiles;
        r.step = paged ? p.H_KV : 1;
    } else {
        // Workgroups reach the XCDs in turn.  Where the pairs divide among them each XCD has its own, one after the other, else
        // the longest workgroups of all pairs come first.  The second workgroups of the CUs are in reverse, so that long and
        // short ones share a CU.
        int pair;
        const int i = int(blockIdx.x), per_xcd = p.pairs * p.W >> 3;
        if ((p.pairs & 7) == 0) {
            int j = i >> 3;
            const int cus = p.round_slots >> 3, both = per_xcd < 2 * cus ? per_xcd : 2 * cus;
            if (AttendCfg<D>::WAVES == 2 && j >= cus && j < both) j = cus + both - 1 - j;
            pair = (j / p.W) * 8 + (i & 7);
            x = p.W - 1 - j % p.W;
        } else {
            int j = i;
            const int all = p.pairs * p.W, both = all < 2 * p.round_slots ? all : 2 * p.round_slots;
            if (AttendCfg<D>::WAVES == 2 && j >= p.round_slots && j < both) j = p.round_slots + both - 1 - j;
            x = p.W - 1 - j / p.pairs;
            pair = j % p.pairs;
        }
        b = (p.pair0 + pair) / p.H_KV;
        hkv = (p.pair0 + pair) % p.H_KV;
        r.at = pair * p.tiles;
        r.step = 1;
    }
    const int NQ = r.NQ, units = ((NQ + 31) >> 5) * p.G;
    const int unit_raw = 4 * x + w;
    r.live = unit_raw < units;
    const int unit = r.live ? unit_raw : units - 1;
    const int hq = hkv * p.G + unit % p.G;
    r.row0 = 32 * (unit / p.G);
    r.q0 = paged ? (int64_t(q_first) * p.H_Q + hq) * D : (int64_t(b) * p.H_Q + hq) * NQ * D;
    r.q_stride = paged ? p.H_Q * D : D;
    const int last_unit = 4 * x + 3 < units - 1 ? 4 * x + 3 : units - 1;
    int wg_maxpos = 32 * (last_unit / p.G) + 31;
    wg_maxpos = qoff + (wg_maxpos < NQ - 1 ? wg_maxpos : NQ - 1);
    const int my_maxpos = qoff + (r.row0 + 31 < NQ - 1 ? r.row0 + 31 : NQ - 1);
    const int all_tiles = (NKV + TT - 1) >> TS;
    int ntiles = all_tiles, my_tiles = all_tiles, full = NKV >> TS;
    if (p.causal) {
        ntiles = (wg_maxpos >> TS) + 1 < all_tiles ? (wg_maxpos >> TS) + 1 : all_tiles;
        my_tiles = (my_maxpos >> TS) + 1 < all_tiles ? (my_maxpos >> TS) + 1 : all_tiles;
        full = (qoff + r.row0 + 1) >> TS < full ? (qoff + r.row0 + 1) >> TS : full;
    }
    int first = 0, end = ntiles;
    if (PLANNED && r.pieces > 1) {      // (less than 2^31: at most four times as many pieces as CUs, of 2^18 tiles)
        first = ntiles * piece / r.pieces;
        end = ntiles * (piece + 1) / r.pieces;
    }
    my_tiles = my_tiles < end ? my_tiles : end;
    r.at += first * r.step;
    r.ntiles = end - first;
    r.my_tiles = r.live && my_tiles > first ? my_tiles - first : 0;
    r.full = full - first;
    r.pos0 = qoff + r.row0 - first * TT;
    r.NKV = NKV - first * TT;
    return r;
}

// A workgroup is 4 wavefronts of 32 positions of one query head each, over the tiles from the first on, double buffered (at 256
// coordinates four times), one barrier a tile.
// What bounds it: power.  v_mfma_f32_32x32x16_f16 alone, on random operands on all CUs, runs at 22.7 ns an instruction and SIMD (the
// clock falls to 1.65 GHz; 14.8 ns on constant ones), which is 1.45 us for the 64 of 256 rows x 64 tokens of 128 coordinates; this loop
// takes 2.06 us.  On a full chip its schedules (products and weights in turn, or the steps below; 4 or 8 wavefronts; 2 or 4
// buffers) differ by 1 %; without exponentials it is 7 % faster, without operand reads 6 %, without the tiles' way into LDS 9 %.
// On a chip that is not full the steps below are 8 % faster (64 workgroups over 8192 keys 164 and 151 us).  64 rows a wavefront (one a
// SIMD, half of the operand reads) 2270 -> 2500 us at 4 x 32 heads x 8192 tokens.
template <int D, int DT, bool PLANNED, bool BIG>
__device__ __forceinline__ void attend_rows(const AttendParams& p, const Rows& rows, uint8_t* lds) {
    using C = TileCfg<D>;
    constexpr int NKS = C::NKS, NOB = C::NOB, TT = C::TT, HT = TT / 32, NBUF = AttendCfg<D>::NBUF;
    const int lane = threadIdx.x & 63, m32 = lane & 31, hf = lane >> 5;
    const int pos0 = rows.pos0, w = rows.w, ntiles = rows.ntiles, my_tiles = rows.my_tiles, full = rows.full, NQ = rows.NQ, NKV = rows.NKV;

    // ---- tiles: every wavefront asks for its quarter, straight into LDS -------------------------------------
    const uint8_t* img = p.images + int64_t(rows.at) * C::TILE;
    constexpr int REQ = C::SIDE / 4096;                                  // requests of a wavefront for one side of a tile
    // (a buffer resource, not global addresses: behind a global_load_lds the compiler waits for all outstanding LDS reads at
    // every use of one, as it would behind a flat access)
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(img), 0, ntiles * rows.step * C::TILE, 0x00027000);
    auto request = [&](int tile, int side) __attribute__((always_inline)) {
        const int src = tile * rows.step * C::TILE + side * C::SIDE + w * (REQ * 1024);
        uint8_t* dst = lds + (tile & (NBUF - 1)) * C::TILE + side * C::SIDE + w * (REQ * 1024);
#pragma unroll
        for (int i = 0; i < REQ; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(dst + i * 1024), 16, lane * 16,
                                                     src + i * 1024, 0, 0);
    };

    // ---- the query rows, exact in fp16 up to a power of two -------------------------------------------------
    half8 qb[NKS];
    float krow;
    {
        const int row = rows.row0 + m32 < NQ ? rows.row0 + m32 : NQ - 1;
        const uint16_t* qrow = p.q + (rows.q0 + int64_t(row) * rows.q_stride);
        uint4v raw[NKS];
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) raw[ks] = *reinterpret_cast<const uint4v*>(qrow + 16 * ks + 8 * hf);
        float mx = 0.0f;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                mx = __builtin_fmaxf(mx, __builtin_fmaxf(__builtin_fabsf(load_elem<DT>(uint16_t(raw[ks][i] & 0xffffu))),
                                                         __builtin_fabsf(load_elem<DT>(uint16_t(raw[ks][i] >> 16)))));
        const int ex = row_exponent(mx);
        krow = p.scale_log2e * pow2(ex);
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                qb[ks][2 * i] = _Float16(load_elem<DT>(uint16_t(raw[ks][i] & 0xffffu)) * pow2(-ex));
                qb[ks][2 * i + 1] = _Float16(load_elem<DT>(uint16_t(raw[ks][i] >> 16)) * pow2(-ex));
            }
    }
    // ---- running state --------------------------------------------------------------------------------------
    float16v O[NOB], S;                            // S: the scores of the next step
    uint4v P[2];                                   // the weights of the last one
    float m_run = -__builtin_inff(), l_run = 0.0f, alpha = 1.0f;
#pragma unroll
    for (int ob = 0; ob < NOB; ++ob)
#pragma unroll
        for (int e = 0; e < 16; ++e) O[ob][e] = 0.0f;

    // Step h is 32 tokens: half a tile, at 256 coordinates a tile.
    auto k_at = [&](int h) __attribute__((always_inline)) { return lds + ((h / HT) & (NBUF - 1)) * C::TILE + (h % HT) * (NKS * 1024) + 16 * lane; };
    auto v_at = [&](int h) __attribute__((always_inline)) {
        return lds + ((h / HT) & (NBUF - 1)) * C::TILE + C::SIDE + (h % HT) * (2 * NOB * 1024) + 16 * lane;
    };
    auto operand = [](const uint8_t* at, int i) __attribute__((always_inline)) { return *reinterpret_cast<const half8*>(at + i * 1024); };
    auto scores = [&](int h) __attribute__((always_inline)) {
        float16v s = {};
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(operand(k_at(h), ks), qb[ks], s, 0, 0, 0);
        return s;
    };
    auto output = [&](int h) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int ob = 0; ob < NOB; ++ob)
                O[ob] = __builtin_amdgcn_mfma_f32_32x32x16_f16(operand(v_at(h), u * NOB + ob), __builtin_bit_cast(half8, P[u]), O[ob], 0, 0, 0);
    };
    auto rescale = [&]() __attribute__((always_inline)) {
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int ob = 0; ob < NOB; ++ob)
#pragma unroll
                for (int e = 0; e < 16; ++e) O[ob][e] *= alpha;
        }
    };
    auto hide = [&](int h) __attribute__((always_inline)) {              // scores of keys that the rows do not see
        int lim = NKV - 1;
        if (p.causal && pos0 + m32 < lim) lim = pos0 + m32;
        lim -= 32 * h;
#pragma unroll
        for (int e = 0; e < 16; ++e)
            if (8 * (e >> 2) + 4 * hf + (e & 3) > lim) S[e] = -__builtin_inff();
    };
    // The reference of the weights moves only when a score would lead it by more than 2^4: the weights stay below 16 and the
    // rescale of the accumulators is rare.
    auto move_reference = [&](float cand) __attribute__((always_inline)) {
        cand = max_xor32(cand);
        const float mnew = cand > m_run + 4.0f ? cand : m_run;
        const float ms = mnew == -__builtin_inff() ? 0.0f : mnew;
        alpha = __builtin_amdgcn_exp2f(m_run - ms);
        m_run = mnew;
        return ms;
    };
    auto largest = [&]() __attribute__((always_inline)) {
        float mx = S[0];
#pragma unroll
        for (int e = 1; e < 16; ++e) mx = __builtin_fmaxf(mx, S[e]);
        return mx * krow;
    };
    const half2v ones = {_Float16(1.0f), _Float16(1.0f)};
    // The weights of step h from the scores in S, on their own.
    auto weights = [&](int h) __attribute__((always_inline)) {
        const int64_t block = (int64_t(rows.at) + (h / HT) * rows.step) * 2 * HT + h % HT;        // of the keys; + HT: of the values
        auto exps_of = [&](int side, int q) __attribute__((always_inline)) {
            const int4v none = {0, 0, 0, 0};
            return BIG && p.flags[block + side * HT] != 0
                       ? *reinterpret_cast<const int4v*>(p.exps + (block + side * HT) * 32 + 8 * q + 4 * hf) : none;
        };
        if constexpr (BIG) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int4v e = exps_of(0, q);
#pragma unroll
                for (int c = 0; c < 4; ++c) S[4 * q + c] = __builtin_ldexpf(S[4 * q + c], e[c]);
            }
        }
        hide(h);
        float cand = -__builtin_inff();
        if constexpr (BIG) {
            // a value row stored divided by 2^e gets its weight multiplied by 2^e: the reference is taken over score + e, so
            // that these weights stay below 16 as well
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int4v e = exps_of(1, q);
#pragma unroll
                for (int c = 0; c < 4; ++c) cand = __builtin_fmaxf(cand, __builtin_fmaf(S[4 * q + c], krow, float(e[c])));
            }
        } else {
            cand = largest();
        }
        const float ms = move_reference(cand);
        float ps = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float pe[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) pe[c] = __builtin_amdgcn_exp2f(__builtin_fmaf(S[4 * q + c], krow, -ms));
            if constexpr (BIG) {
                const int4v e = exps_of(1, q);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    ps += pe[c];
                    pe[c] = __builtin_ldexpf(pe[c], e[c]);
                }
            }
#pragma unroll
            for (int c = 0; c < 4; c += 2) {
                const uint32_t two = pack_weights<D>(pe[c], pe[c + 1]);
                if constexpr (!BIG) ps = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2v, two), ones, ps, false);
                P[q >> 1][2 * (q & 1) + (c >> 1)] = two;
            }
        }
        l_run = __builtin_fmaf(l_run, alpha, ps);
    };
    // Step h: the scores of step h + 1, the weights of step h and the output of step h - 1, which do not wait for one another.
    // One product, one operand read and a part of the weights a slot, in this order (the compiler left alone reads an operand
    // right in front of its product); the operands of the scores are asked for before the largest score is looked for.
    auto step = [&](int h, auto masked) __attribute__((always_inline)) {
        constexpr int SLOTS = NKS + 2 * NOB;
        const uint8_t *kt = k_at(h + 1), *vt = v_at(h - 1);
        half8 k[NKS], v[2 * NOB];
#pragma unroll
        for (int i = 0; i < NKS; ++i) k[i] = operand(kt, i);
#pragma unroll
        for (int i = 0; i < NOB; ++i) v[i] = operand(vt, i);
        if constexpr (decltype(masked)::value) hide(h);
        const float ms = move_reference(largest());
        __builtin_amdgcn_sched_barrier(0);
        float16v next = {};
        uint4v pw[2];
        float wa = 0.0f, wb = 0.0f, ps = 0.0f;
        auto finish = [&](int j) __attribute__((always_inline)) {        // pair j of the weights
            const uint32_t two = pack_weights<D>(wa, wb);
            pw[j >> 2][j & 3] = two;
            // the denominator sums the weights as the products see them
            ps = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2v, two), ones, ps, false);
        };
#pragma unroll
        for (int n = 0; n < SLOTS; ++n) {
            if (n < NKS) {
                next = __builtin_amdgcn_mfma_f32_32x32x16_f16(k[n], qb[n], next, 0, 0, 0);
            } else {
                const int ob = (n - NKS) % NOB, u = (n - NKS) / NOB;
                O[ob] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[n - NKS], __builtin_bit_cast(half8, P[u]), O[ob], 0, 0, 0);
            }
            if (n < NOB) v[NOB + n] = operand(vt, NOB + n);
#pragma unroll
            for (int e = n * 16 / SLOTS; e < (n + 1) * 16 / SLOTS; ++e) {
                if ((e & 1) == 0 && e > 0) finish(e / 2 - 1);
                (e & 1 ? wb : wa) = __builtin_amdgcn_exp2f(__builtin_fmaf(S[e], krow, -ms));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        finish(7);
        l_run = __builtin_fmaf(l_run, alpha, ps);
        S = next;
        P[0] = pw[0];
        P[1] = pw[1];
        asm volatile("" : "+v"(P[0]), "+v"(P[1]));                       // (made here, not behind the branch)
        rescale();
    };
    auto step_big = [&](int h) __attribute__((always_inline)) {
        const float16v next = scores(h + 1);
        output(h - 1);
        weights(h);
        rescale();
        S = next;
    };

    // ---- tiles ----------------------------------------------------------------------------------------------
    // Iteration i runs the steps up to the first of tile i + 1: it needs the keys of tile i + KA and the values of tile i,
    // and all wavefronts are done with the keys of tile i and the values of tile i - 1.
    constexpr int KA = HT == 1 ? 2 : 1;
    auto meet = [&](int i) __attribute__((always_inline)) {
        if (NBUF > KA + 1 && i - 1 + NBUF < ntiles) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * REQ * (NBUF - 1 - KA)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (i + NBUF < ntiles) request(i + NBUF, 0);
        if (i - 1 + NBUF < ntiles) request(i - 1 + NBUF, 1);
    };
#pragma unroll
    for (int t = 0; t < NBUF; ++t) {
        if (t < ntiles) request(t, 0);
        if (t < ntiles && t < NBUF - 1) request(t, 1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int i = 0;
    if (my_tiles > 0) {
        S = scores(0);
        const float16v next = scores(1);
        weights(0);
        S = next;
    }
    if constexpr (!BIG) {
        for (; i + 1 < full && i + 1 < my_tiles; ++i) {
            meet(i);
            step(HT * i + 1, std::false_type{});
            if (HT == 2) step(2 * i + 2, std::false_type{});
        }
    }
    for (; i + 1 < my_tiles; ++i) {
        meet(i);
        if constexpr (BIG) {
            step_big(HT * i + 1);
            if (HT == 2) step_big(2 * i + 2);
        } else {
            step(HT * i + 1, std::true_type{});
            if (HT == 2) step(2 * i + 2, std::true_type{});
        }
    }
    if (i < my_tiles) {
        meet(i);
        output(HT * i);
        if (HT == 2) {
            weights(2 * i + 1);
            rescale();
            output(2 * i + 1);
        }
        ++i;
    }
    for (; i < ntiles; ++i) meet(i);                                     // tiles only the other wavefronts need

    const float l_tot = l_run + xor_shuffle(l_run, 32);
    if (!rows.live || rows.row0 + m32 >= NQ) return;
    // ---- a piece: the rows as they lie in the registers, for the combine launch ------------------------------
    if (PLANNED && rows.pieces > 1) {
        float* part = p.part + (int64_t(rows.slot) * 4 + w) * C::UNIT;
#pragma unroll
        for (int ob = 0; ob < NOB; ++ob)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<float4v*>(part + ((4 * ob + q) * 64 + lane) * 4) =
                    float4v{O[ob][4 * q], O[ob][4 * q + 1], O[ob][4 * q + 2], O[ob][4 * q + 3]};
        part[32 * D + lane] = hf == 0 ? m_run : l_tot;
        return;
    }
    // ---- normalise, store: register e of half hf is coordinate 32 ob + 16 (e / 8) + 8 hf + e % 8 --------------
    const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    uint16_t* orow = p.out + (rows.q0 + int64_t(rows.row0 + m32) * rows.q_stride);
#pragma unroll
    for (int ob = 0; ob < NOB; ++ob)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            uint4v v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = round_pair<DT>(O[ob][8 * u + 2 * e] * inv, O[ob][8 * u + 2 * e + 1] * inv);
            uint16_t* dst = orow + 32 * ob + 16 * u + 8 * hf;
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

template <int D, int DT, bool PLANNED>
__global__ __launch_bounds__(256, AttendCfg<D>::WAVES) void attend_expanded_kernel(const AttendParams p) {
    extern __shared__ __attribute__((aligned(256))) uint8_t lds[];      // NBUF tiles
    const Rows rows = rows_of<D, PLANNED>(p);
    if (PLANNED && rows.none) return;                                              // (the grid is sized for the most work possible)
    // Tiles with rows of long norms take a loop of their own, all of it: where the two met again the compiler spilled 80
    // registers at 128 coordinates.
    constexpr int PER = 2 * TileCfg<D>::NTB;
    typedef int flags_of_tile __attribute__((ext_vector_type(PER)));
    const flags_of_tile* flags = reinterpret_cast<const flags_of_tile*>(p.flags) + rows.at;
    int longs = 0;
    for (int t = threadIdx.x & 63; t < rows.ntiles; t += kWave) {
        const flags_of_tile f = flags[t * rows.step];
#pragma unroll
        for (int i = 0; i < PER; ++i) longs |= f[i];
    }
    if (__any(longs != 0)) attend_rows<D, DT, PLANNED, true>(p, rows, lds);
    else attend_rows<D, DT, PLANNED, false>(p, rows, lds);
}

// Rows of workgroups in several pieces: the pieces' rows weighted by 2^(m - max m), summed and normalised.  A workgroup takes a unit
// (32 rows, a lane a row and half of its coordinates, as they were left).
template <int D, int DT>
__global__ __launch_bounds__(256) void combine_expanded_kernel(const AttendParams p) {
    using C = TileCfg<D>;
    const int lane = threadIdx.x & 63, m32 = lane & 31, hf = lane >> 5, wave = threadIdx.x >> 6;
    const int u = int(blockIdx.x) & 3, hkv = (int(blockIdx.x) >> 2) % p.H_KV, entry = (int(blockIdx.x) >> 2) / p.H_KV;
    if (entry >= p.plan.counts[1]) return;
    const WorkPiece wp = p.plan.splits[entry];
    const int units = ((wp.NQ + 31) >> 5) * p.G, unit = 4 * wp.x + u;
    if (unit >= units) return;
    const int row = 32 * (unit / p.G) + m32, hq = hkv * p.G + unit % p.G;
    if (row >= wp.NQ) return;
    const int64_t next = int64_t(p.H_KV) * 4 * C::UNIT;                 // floats from a piece to the next
    const float* part = p.part + (int64_t(wp.slot) * p.H_KV + hkv) * 4 * C::UNIT + u * C::UNIT;
    float top = -__builtin_inff();
    for (int k = 0; k < wp.pieces; ++k) top = __builtin_fmaxf(top, part[k * next + 32 * D + m32]);
    float den = 0.0f;
    for (int k = 0; k < wp.pieces; ++k) {
        const float m = part[k * next + 32 * D + m32], l = part[k * next + 32 * D + 32 + m32];
        den = __builtin_fmaf(l, piece_weight(m, l, top), den);
    }
    const float inv = inverse_sum(den);
    uint16_t* orow = p.out + (p.paged ? (int64_t(wp.q_first + row) * p.H_Q + hq) * D : ((int64_t(wp.seq) * p.H_Q + hq) * wp.NQ + row) * D);
    for (int ob = wave; ob < C::NOB; ob += 4) {
        float sum[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) sum[e] = 0.0f;
        for (int k = 0; k < wp.pieces; ++k) {
            const float wk = piece_weight(part[k * next + 32 * D + m32], part[k * next + 32 * D + 32 + m32], top);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4v v = *reinterpret_cast<const float4v*>(part + k * next + ((4 * ob + q) * 64 + lane) * 4);
#pragma unroll
                for (int c = 0; c < 4; ++c) sum[4 * q + c] = __builtin_fmaf(v[c], wk, sum[4 * q + c]);
            }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            uint4v v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = round_pair<DT>(sum[8 * h + 2 * e] * inv, sum[8 * h + 2 * e + 1] * inv);
            uint16_t* dst = orow + 32 * ob + 16 * h + 8 * hf;
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
}

template <int D>
int launch_expanded(ExpandParams e, AttendParams a, int dtype, const ExpandedPlan& ep, int64_t pairs, hipStream_t s) {
    using C = TileCfg<D>;
    const size_t elds = 65536 + 2 * C::RTERM, alds = AttendCfg<D>::NBUF * C::TILE;
    const int64_t cus = fq_host::device_cu_count();
    // items of 32 tokens where ones of 64 would leave wavefronts without any
    const bool small = D != 256 && (a.paged ? int64_t(ep.tiles) * a.H_KV : pairs * ep.tiles) * 2 < 8 * cus;
    const bool paged = a.paged, planned = e.planned;
    constexpr int TB = C::NTB;
    auto expand = small ? (paged ? tq4_expand_kernel<D, 1, true, true> : (planned ? tq4_expand_kernel<D, 1, false, true> : tq4_expand_kernel<D, 1, false, false>))
                        : (paged ? tq4_expand_kernel<D, TB, true, true> : (planned ? tq4_expand_kernel<D, TB, false, true> : tq4_expand_kernel<D, TB, false, false>));
    auto attend = dtype == FQ_F16 ? (planned ? attend_expanded_kernel<D, FQ_F16, true> : attend_expanded_kernel<D, FQ_F16, false>)
                                  : (planned ? attend_expanded_kernel<D, FQ_BF16, true> : attend_expanded_kernel<D, FQ_BF16, false>);
    auto combine = dtype == FQ_F16 ? combine_expanded_kernel<D, FQ_F16> : combine_expanded_kernel<D, FQ_BF16>;
    if (!fq_host::lds_limit_raised(reinterpret_cast<const void*>(expand), elds)) return FQ_ERR_LAUNCH;
    if (!fq_host::lds_limit_raised(reinterpret_cast<const void*>(attend), alds)) return FQ_ERR_LAUNCH;
    for (int64_t first = 0; first < pairs; first += ep.per_chunk) {
        e.pair0 = a.pair0 = int(first);
        e.pairs = a.pairs = int(pairs - first < ep.per_chunk ? pairs - first : ep.per_chunk);
        const int64_t items = (a.paged ? int64_t(ep.tiles) * a.H_KV : int64_t(e.pairs) * ep.tiles) * 2 * (small ? 2 : 1);
        int64_t grid = items < cus / C::ROUNDS ? items : cus / C::ROUNDS;
        if (e.planned) grid = grid + 1 < cus / C::ROUNDS ? grid + 1 : cus / C::ROUNDS;
        hipLaunchKernelGGL(expand, dim3(unsigned(grid), C::ROUNDS), dim3(512), elds, s, e);
        int st = fq_host::check_launch();
        if (st != FQ_OK) return st;
        const int64_t wgs = e.planned ? int64_t(a.plan.max_items) * a.H_KV : int64_t(a.pairs) * a.W;
        hipLaunchKernelGGL(attend, dim3(unsigned(wgs)), dim3(256), alds, s, a);
        st = fq_host::check_launch();
        if (st != FQ_OK) return st;
        if (e.planned && a.plan.max_slots > 0) {
            hipLaunchKernelGGL(combine, dim3(unsigned(a.plan.max_slots / 2) * unsigned(a.H_KV) * 4), dim3(256), 0, s, a);
            st = fq_host::check_launch();
            if (st != FQ_OK) return st;
        }
    }
    return FQ_OK;
}

}  // namespace

int launch_attention_expanded(ExpandParams e, AttendParams a, const ExpandedPlan& ep, int D, int dtype, void* workspace, void* stream) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    e.tiles = a.tiles = ep.tiles;
    e.keys = ep.keys;
    e.images = ws;
    e.flags = reinterpret_cast<int*>(ws + ep.images);
    e.exps = reinterpret_cast<int*>(ws + ep.images + ep.flags);
    a.images = e.images; a.flags = e.flags; a.exps = e.exps;
    a.W = ((a.N_Q + 31) / 32 * a.G + 3) / 4;
    a.round_slots = fq_host::device_cu_count();
    e.planned = ep.max_items > 0;
    e.H_KV = a.H_KV; e.G = a.G; e.N_Q = a.N_Q; e.causal = a.causal;
    if (e.planned) {
        WorkPlan w{};
        uint8_t* at = ws + ep.images + ep.flags + ep.exps;
        w.counts = reinterpret_cast<int*>(at);
        w.items = reinterpret_cast<WorkPiece*>(at + 256);
        w.splits = w.items + ep.max_items;
        w.max_items = ep.max_items; w.max_slots = ep.max_slots; w.cus = ep.cus; w.cu_slots = ep.cu_slots;
        e.plan = a.plan = w;
        a.part = reinterpret_cast<float*>(at + ep.plan);
    }
    const int64_t pairs = a.paged ? 1 : int64_t(e.num_seqs) * a.H_KV;
    if (D == 64) return launch_expanded<64>(e, a, dtype, ep, pairs, s);
    if (D == 128) return launch_expanded<128>(e, a, dtype, ep, pairs, s);
    return launch_expanded<256>(e, a, dtype, ep, pairs, s);
}

}  // namespace fq
