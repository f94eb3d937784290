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

// An item is TBI blocks of 32 tokens of the keys or the values of a pair, on one wavefront from the packed rows to the image, with no
// barrier: lookups (pair table as in the other kernels) into matrix operands, the products with both terms of the matrix out of
// LDS (two fp16 terms of 256 R: 2^-22 of its largest entry), the norm in float32, one rounding.  A lane's half row is contiguous
// (the contraction index is permuted on both sides), its result registers are whole operands of the image.  At 256 coordinates
// the matrix is 256 KB and blockIdx.y has a quarter of the columns.
// Bound by the stores where there are many tiles (4 x 8 heads x 8192 tokens of 128 45 us, 134 MB), by the start (5.3 us: matrix
// and tables) and one item's chain where there are few: 8 heads x 65 tokens 7.6 us.  Stores that stay out of the L2 (nontemporal)
// 18.9 -> 15.6 us at 128 pairs x 300 tokens: else they are written back at the end of the launch.
template <int D, int TBI>
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
    const int items = p.pairs * p.tiles * 2 * IPT;
    const int stride = int(gridDim.x);

    uint4v raw[NTB][DW / 4];
    float nrm[NTB];
    auto issue = [&](int item_raw) {
        const int item = item_raw < items ? item_raw : items - 1;
        const int side = item & 1, part = (item >> 1) % IPT, at = (item >> 1) / IPT, tile = at % p.tiles, pair = p.pair0 + at / p.tiles;
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
    issue(item);
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

// What a wavefront has to do: 32 positions of one query head, and the tiles they see.
struct Rows {
    int pair, b, hq, pos0, w;
    int ntiles, my_tiles, full;         // of the workgroup; of this wavefront; that hide nothing from its rows
    bool live;
};

template <int D>
__device__ __forceinline__ Rows rows_of(const AttendParams& p) {
    using C = TileCfg<D>;
    constexpr int TT = C::TT, TS = C::TS;
    const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    // Workgroups reach the XCDs in turn.  Where the pairs divide among them each XCD has its own, one after the other, else the
    // longest workgroups of all pairs come first.  The second workgroups of the CUs are in reverse, so that long and short ones
    // share a CU.
    int pair, x;
    {
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
    }
    const int at = p.pair0 + pair, b = at / p.H_KV, hkv = at % p.H_KV;
    const int NQ = p.N_Q, NKV = p.N_KV;
    const int units = ((NQ + 31) >> 5) * p.G;
    const int unit_raw = 4 * x + w;
    const bool live = unit_raw < units;
    const int unit = live ? unit_raw : units - 1;
    const int hq = hkv * p.G + unit % p.G, pos0 = 32 * (unit / p.G);
    const int last_unit = 4 * x + 3 < units - 1 ? 4 * x + 3 : units - 1;
    int wg_maxpos = 32 * (last_unit / p.G) + 31;
    wg_maxpos = wg_maxpos < NQ - 1 ? wg_maxpos : NQ - 1;
    const int my_maxpos = pos0 + 31 < NQ - 1 ? pos0 + 31 : NQ - 1;
    const int all_tiles = (NKV + TT - 1) >> TS;
    int ntiles = all_tiles, my_tiles = all_tiles, full = NKV >> TS;     // `full`: tiles that hide nothing from these rows
    if (p.causal) {
        ntiles = (wg_maxpos >> TS) + 1 < all_tiles ? (wg_maxpos >> TS) + 1 : all_tiles;
        my_tiles = (my_maxpos >> TS) + 1 < all_tiles ? (my_maxpos >> TS) + 1 : all_tiles;
        full = (pos0 + 1) >> TS < full ? (pos0 + 1) >> TS : full;
    }
    if (!live) my_tiles = 0;
    return Rows{pair, b, hq, pos0, w, ntiles, my_tiles, full, live};
}

// A workgroup is 4 wavefronts of 32 positions of one query head each, over the tiles from the first on, double buffered (at 256
// coordinates four times), one barrier a tile.
// What bounds it: power.  v_mfma_f32_32x32x16_f16 alone, on random operands on all CUs, runs at 22.7 ns an instruction and SIMD (the
// clock falls to 1.65 GHz; 14.8 ns on constant ones), which is 1.45 us for the 64 of 256 rows x 64 tokens of 128 coordinates; this loop
// takes 2.06 us.  On a full chip its schedules (products and weights in turn, or the steps below; 4 or 8 wavefronts; 2 or 4
// buffers) differ by 1 %; without exponentials it is 7 % faster, without operand reads 6 %, without the tiles' way into LDS 9 %.
// On a chip that is not full the steps below are 8 % faster (64 workgroups over 8192 keys 164 and 151 us).  64 rows a wavefront (one a
// SIMD, half of the operand reads) 2270 -> 2500 us at 4 x 32 heads x 8192 tokens.
template <int D, int DT, bool BIG>
__device__ __forceinline__ void attend_rows(const AttendParams& p, const Rows& rows, uint8_t* lds) {
    using C = TileCfg<D>;
    constexpr int NKS = C::NKS, NOB = C::NOB, TT = C::TT, HT = TT / 32, NBUF = AttendCfg<D>::NBUF;
    const int lane = threadIdx.x & 63, m32 = lane & 31, hf = lane >> 5;
    const int pair = rows.pair, b = rows.b, hq = rows.hq, pos0 = rows.pos0, w = rows.w;
    const int ntiles = rows.ntiles, my_tiles = rows.my_tiles, full = rows.full;
    const int NQ = p.N_Q, NKV = p.N_KV;

    // ---- tiles: every wavefront asks for its quarter, straight into LDS -------------------------------------
    const uint8_t* img = p.images + int64_t(pair) * p.tiles * C::TILE;
    constexpr int REQ = C::SIDE / 4096;                                  // requests of a wavefront for one side of a tile
    // (a buffer resource, not global addresses: behind a global_load_lds the compiler waits for all outstanding LDS reads at
    // every use of one, as it would behind a flat access)
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(img), 0, p.tiles * C::TILE, 0x00027000);
    auto request = [&](int tile, int side) __attribute__((always_inline)) {
        const int src = tile * C::TILE + side * C::SIDE + w * (REQ * 1024);
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
        const int pos = pos0 + m32 < NQ ? pos0 + m32 : NQ - 1;
        const uint16_t* qrow = p.q + ((int64_t(b) * p.H_Q + hq) * NQ + pos) * D;
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
        const int64_t block = (int64_t(pair) * p.tiles + h / HT) * 2 * HT + h % HT;        // of the keys; + HT: of the values
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

    // ---- normalise, store: register e of half hf is coordinate 32 ob + 16 (e / 8) + 8 hf + e % 8 --------------
    const float l_tot = l_run + xor_shuffle(l_run, 32);
    const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    if (!rows.live || pos0 + m32 >= NQ) return;
    uint16_t* orow = p.out + ((int64_t(b) * p.H_Q + hq) * NQ + pos0 + m32) * D;
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

template <int D, int DT>
__global__ __launch_bounds__(256, AttendCfg<D>::WAVES) void attend_expanded_kernel(const AttendParams p) {
    extern __shared__ __attribute__((aligned(256))) uint8_t lds[];      // NBUF tiles
    const Rows rows = rows_of<D>(p);
    // Tiles with rows of long norms take a loop of their own, all of it: where the two met again the compiler spilled 80
    // registers at 128 coordinates.
    constexpr int PER = 2 * TileCfg<D>::NTB;
    const int* flags = p.flags + int64_t(rows.pair) * p.tiles * PER;
    int longs = 0;
    for (int t = 2 * (threadIdx.x & 63); t < PER * rows.ntiles; t += 2 * kWave) longs |= flags[t] | flags[t + 1];
    if (__any(longs != 0)) attend_rows<D, DT, true>(p, rows, lds);
    else attend_rows<D, DT, false>(p, rows, lds);
}

template <int D>
int launch_expanded(ExpandParams e, AttendParams a, int dtype, int64_t pairs, int64_t per_chunk, hipStream_t s) {
    using C = TileCfg<D>;
    const size_t elds = 65536 + 2 * C::RTERM, alds = AttendCfg<D>::NBUF * C::TILE;
    // items of 32 tokens where ones of 64 would leave wavefronts without any
    const bool small = D != 256 && pairs * e.tiles * 2 < 8 * int64_t(fq_host::device_cu_count());
    auto expand = small || D == 256 ? tq4_expand_kernel<D, 1> : tq4_expand_kernel<D, C::NTB>;
    if (!fq_host::lds_limit_raised(reinterpret_cast<const void*>(expand), elds)) return FQ_ERR_LAUNCH;
    auto attend = dtype == FQ_F16 ? attend_expanded_kernel<D, FQ_F16> : attend_expanded_kernel<D, FQ_BF16>;
    if (!fq_host::lds_limit_raised(reinterpret_cast<const void*>(attend), alds)) return FQ_ERR_LAUNCH;
    for (int64_t first = 0; first < pairs; first += per_chunk) {
        e.pair0 = a.pair0 = int(first);
        e.pairs = a.pairs = int(pairs - first < per_chunk ? pairs - first : per_chunk);
        const int64_t items = int64_t(e.pairs) * e.tiles * 2 * (small ? 2 : 1);
        const int64_t cus = fq_host::device_cu_count() / C::ROUNDS;
        hipLaunchKernelGGL(expand, dim3(unsigned(items < cus ? items : cus), C::ROUNDS), dim3(512), elds, s, e);
        int st = fq_host::check_launch();
        if (st != FQ_OK) return st;
        hipLaunchKernelGGL(attend, dim3(unsigned(a.pairs) * unsigned(a.W)), dim3(256), alds, s, a);
        st = fq_host::check_launch();
        if (st != FQ_OK) return st;
    }
    return FQ_OK;
}

}  // namespace

int launch_attention_expanded(const ExpandParams& e, const AttendParams& a, int D, int dtype, int64_t pairs, int64_t per_chunk,
                              void* stream) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (D == 64) return launch_expanded<64>(e, a, dtype, pairs, per_chunk, s);
    if (D == 128) return launch_expanded<128>(e, a, dtype, pairs, per_chunk, s);
    return launch_expanded<256>(e, a, dtype, pairs, per_chunk, s);
}

}  // namespace fq
