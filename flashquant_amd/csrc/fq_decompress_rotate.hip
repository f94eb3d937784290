// TQ4 decompress with the inverse rotation, one launch, gfx950.
//
// What the serving path does in two steps when it materialises the cache
// (_decompress_cache, src/flashquant/vllm/impl.py:265-318): tq4_decompress to the compute
// dtype (decompress_reference, src/flashquant/kernels/cpu_reference.py:64-94, cast at
// src/flashquant/kernels/decompress.py:80-81), then (x.float() @ rotation).to(dtype)
// (impl.py:309-316).  Per row:
//
//   v_j   = dtype(float32(centroid[idx_j] * norm))          rotated space, two roundings
//   out_i = dtype(sum_j float32(v_j) * R[j][i])             original space
//
// Bytes per row: 4 + D/2 in, 2 D out: the kernel is bound by HBM like the plain decompress,
// provided the contraction stays in the shadow of the memory traffic.  The v_j are 16-bit
// values by construction, so they go to the 32x32x16 MFMA of their own type exactly; R is
// stationary in registers as the A operand in two 16-bit terms (bf16: R = t0 + t1 to 2^-17,
// fp16: R = hi + lo / 4096 to 2^-22), which is far below the 2^-9 / 2^-12 rounding of the
// result.  A tile of 64 rows is dequantised into LDS (the B operand), each wavefront produces
// 32 output coordinates of every row, a lane ends with 16 consecutive coordinates of one row
// (the MFMA row index is permuted on the R side), and the rows leave through LDS in full
// 16-byte-per-lane spans.

#include "fq_common.hpp"

namespace fq {

namespace {

// LONG: see launch_decompress_rotate
template <int D, bool LONG>
struct DecRotCfg {
    static constexpr int NK = D / 16;                  // MFMA k-steps
    static constexpr int CB = D / 32;                  // 32-coordinate output blocks
    static constexpr int WAVES = CB < 4 ? 4 : CB;
    static constexpr int THREADS = WAVES * kWave;
    static constexpr int TT = D == 256 && !LONG ? 32 : 64;     // rows per tile
    static constexpr int TB = TT / 32;                 // 32-row blocks per tile
    static constexpr int TB_STEP = WAVES / CB;         // row blocks handled in parallel
    static constexpr int UPR = D / 8;                  // packed dwords (8 coordinates) per row
    static constexpr int UNITS = TT * UPR;             // per tile
    static constexpr int UPT = UNITS / THREADS;        // per thread
    static constexpr int STRIDE = D * 2 + 16;          // bytes per 16-bit row in LDS (padded)
};

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float two_roundings(float c, float n) {
    float p = c * n;                       // float32 product first, as the reference rounds it
    asm("" : "+v"(p));                     // (keeps the compiler from fusing it into the 16-bit conversion;
    return p;                              // not volatile: the products of a row may be scheduled freely)
}

// MFMA row r of a 32-row block <-> output coordinate (within the block) such that accumulator
// register i of lane half h holds coordinate 16 h + i.
__device__ __forceinline__ int row_to_coord(int r) { return 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3); }

// The packed rows of a launch.  Contiguous: `packed` (M, D/2) and `norms` (M,).  CACHE: rows 0 .. M-1 are the keys
// and M .. 2M-1 (tiles from `num_tiles / 2` on) the values of a paged cache's token rows
// [K idx H*D/2 | K norm H*4 | V idx H*D/2 | V norm H*4], read where they are; row (t, h) of either lies
// t * row_bytes + h * D/2 (norm: + 4 h) behind its section's start.  Bound by the launch's start and end (about 8 tiles
// a workgroup) and then by HBM: 24,016 tokens x 8 heads of 128 in bf16 took 89 us as four strided copies of the
// sections and a launch each for keys and values, 40 us this way (124 MB: 25 us at the rate of a plain copy).
struct DecRotSource {
    const uint8_t* packed;
    const float* norms;
    int H;                    // CACHE: KV heads, and
    float inv_H;              // 1 / H
};

template <int D, int DT, bool CACHE, bool LONG>
__global__ __launch_bounds__((DecRotCfg<D, LONG>::THREADS)) void tq4_decompress_rotate_kernel(
    const DecRotSource src, const float* __restrict__ centroids, const float* __restrict__ rotation, int col_major,
    uint16_t* __restrict__ out, uint16_t* __restrict__ out_v, int64_t M, int64_t num_tiles) {
    using C = DecRotCfg<D, LONG>;
    __shared__ __attribute__((aligned(16))) uint8_t xs[2][C::TT * C::STRIDE];   // dequantised rows, 16-bit
    __shared__ __attribute__((aligned(16))) uint8_t os[LONG ? 2 : 1][C::TT * C::STRIDE];     // rotated rows, 16-bit
    __shared__ float lut[16];

    const int tid = threadIdx.x;
    const int wave = tid / kWave, lane = tid % kWave;
    const int n32 = lane % 32, kg = lane / 32;
    const int cb = wave % C::CB, tb0 = wave / C::CB;

    if (tid < 16) lut[tid] = centroids[tid];

    // ---- staging: unit u of a tile = packed dword u % UPR of tile row u / UPR ------------------
    uint32_t word[C::UPT];
    float nrm[C::UPT];
    const int64_t half_tiles = CACHE ? num_tiles / 2 : num_tiles;
    auto issue_loads = [&](int64_t tile) {
        if constexpr (CACHE) {
            // (t0, h0) of the tile's first row once, wave-uniform; a row's own from there with one float32
            // multiply (its numerator stays below 64 + H: exact)
            const bool is_v = tile >= half_tiles;
            const uint32_t row0 = uint32_t(is_v ? tile - half_tiles : tile) * uint32_t(C::TT);
            const uint32_t t0 = row0 / uint32_t(src.H), h0 = row0 - t0 * uint32_t(src.H);
            const int row_bytes = src.H * (D + 8);
            const uint8_t* base = src.packed + int64_t(t0) * row_bytes + (is_v ? src.H * (D / 2 + 4) : 0);
#pragma unroll
            for (int i = 0; i < C::UPT; ++i) {
                const int u = tid + i * C::THREADS;
                const int r = u / C::UPR;
                const bool live = int64_t(row0) + r < M;
                const int local = live ? int(h0) + r : int(h0);
                const int dt = int((float(local) + 0.5f) * src.inv_H), h = local - dt * src.H;
                const uint8_t* row = base + dt * row_bytes;
                word[i] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(row + h * (D / 2)) + u % C::UPR);
                nrm[i] = *reinterpret_cast<const float*>(row + src.H * (D / 2) + 4 * h);
            }
            return;
        }
        const uint32_t* packed = reinterpret_cast<const uint32_t*>(src.packed);
        const float* norms = src.norms;
        if ((tile + 1) * C::TT <= M) {          // uniform: a whole tile needs no per-row conditions
            const uint32_t* first = packed + tile * C::TT * C::UPR;
            const float* nsrc = norms + tile * C::TT;
#pragma unroll
            for (int i = 0; i < C::UPT; ++i) {
                const int u = tid + i * C::THREADS;
                word[i] = __builtin_nontemporal_load(first + u);
                nrm[i] = nsrc[u / C::UPR];
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < C::UPT; ++i) {
            const int u = tid + i * C::THREADS;
            const int64_t row = tile * C::TT + u / C::UPR;
            const bool live = row < M;
            word[i] = live ? __builtin_nontemporal_load(packed + row * C::UPR + u % C::UPR) : 0u;
            nrm[i] = live ? norms[row] : 0.0f;
        }
    };
    // the first tile's rows are asked for before the matrix, whose fetch and split they arrive behind (2 x 12,800 rows
    // of 128 8.1 -> 7.7 us, 2 x 51,200 of 64 8.7 -> 8.3)
    int64_t tile = blockIdx.x;
    if (tile < num_tiles) issue_loads(tile);

    // ---- the matrix rows of this wavefront: A[j][k] = R[k][j], two 16-bit terms ---------------
    constexpr bool kBf16 = DT == FQ_BF16;
    half8 a_hi[kBf16 ? 1 : C::NK], a_lo[kBf16 ? 1 : C::NK];
    bf16x8 a_t[kBf16 ? 2 : 1][kBf16 ? C::NK : 1];
    {
        const int j = 32 * cb + row_to_coord(n32);
#pragma unroll
        for (int ks = 0; ks < C::NK; ++ks) {
            // a lane's eight elements of a k-step are contiguous in a column-major matrix (what a QR factor is);
            // asked for one by one they were 64 requests of 64 lines each in front of the first tile
            float rk[8];
            const int k0 = 16 * ks + 8 * kg;
            if (col_major) {
                typedef float4v float4a __attribute__((aligned(4)));       // the matrix need not be aligned to 16 bytes
                const float4v lo = *reinterpret_cast<const float4a*>(rotation + int64_t(j) * D + k0);
                const float4v hi = *reinterpret_cast<const float4a*>(rotation + int64_t(j) * D + k0 + 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) { rk[e] = lo[e]; rk[4 + e] = hi[e]; }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) rk[e] = rotation[int64_t(k0 + e) * D + j];
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float r = rk[e];
                if constexpr (kBf16) {
                    const uint16_t t0 = float_to_bf16(r);
                    const uint16_t t1 = float_to_bf16(r - bf16_to_float(t0));
                    a_t[0][ks][e] = __builtin_bit_cast(__bf16, t0);
                    a_t[1][ks][e] = __builtin_bit_cast(__bf16, t1);
                } else {
                    const _Float16 hi = _Float16(r);
                    a_hi[ks][e] = hi;
                    a_lo[ks][e] = _Float16((r - float(hi)) * 4096.0f);
                }
            }
        }
    }
    __syncthreads();

    auto stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < C::UPT; ++i) {
            const int u = tid + i * C::THREADS;
            uint32_t h[4];
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const uint32_t byte = (word[i] >> (8 * b)) & 0xffu;
                h[b] = round_pair<DT>(two_roundings(lut[byte >> 4], nrm[i]), two_roundings(lut[byte & 15u], nrm[i]));
            }
            *reinterpret_cast<uint4v*>(&xs[buf][(u / C::UPR) * C::STRIDE + (u % C::UPR) * 16]) = uint4v{h[0], h[1], h[2], h[3]};
        }
    };
    auto store_tile = [&](int64_t any_tile, const uint8_t* rows) {
        constexpr int OC = D / 8;            // 16-byte chunks per output row
        const bool is_v = CACHE && any_tile >= half_tiles;
        const int64_t tile = is_v ? any_tile - half_tiles : any_tile;
        uint16_t* dst = is_v ? out_v : out;
        for (int c = tid; c < C::TT * OC; c += C::THREADS) {
            const int r = c / OC, q = c % OC;
            const int64_t row = tile * C::TT + r;
            if (row < M) {
                const uint4v v = *reinterpret_cast<const uint4v*>(rows + r * C::STRIDE + q * 16);
                __builtin_nontemporal_store(v, reinterpret_cast<uint4v*>(dst + row * D) + q);
            }
        }
    };

    auto rotate_tile = [&](const uint8_t* xs_tile, uint8_t* os_tile) {
        for (int tb = tb0; tb < C::TB; tb += C::TB_STEP) {
            const uint8_t* brow = xs_tile + (32 * tb + n32) * C::STRIDE + kg * 16;
            float16v acc = {};
            float16v acc_lo = {};
            if constexpr (kBf16) {
#pragma unroll
                for (int t = 1; t >= 0; --t)          // the small term first
#pragma unroll
                    for (int ks = 0; ks < C::NK; ++ks) {
                        const bf16x8 b = *reinterpret_cast<const bf16x8*>(brow + ks * 32);
                        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a_t[t][ks], b, acc, 0, 0, 0);
                    }
            } else {
#pragma unroll
                for (int ks = 0; ks < C::NK; ++ks) {
                    const half8 b = *reinterpret_cast<const half8*>(brow + ks * 32);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a_hi[ks], b, acc, 0, 0, 0);
                    acc_lo = __builtin_amdgcn_mfma_f32_32x32x16_f16(a_lo[ks], b, acc_lo, 0, 0, 0);
                }
            }
            uint32_t w[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                float v0 = acc[2 * i], v1 = acc[2 * i + 1];
                if constexpr (!kBf16) {
                    v0 = __builtin_fmaf(acc_lo[2 * i], 1.0f / 4096.0f, v0);
                    v1 = __builtin_fmaf(acc_lo[2 * i + 1], 1.0f / 4096.0f, v1);
                }
                w[i] = round_pair<DT>(v0, v1);
            }
            uint8_t* dst = os_tile + (32 * tb + n32) * C::STRIDE + (32 * cb + 16 * kg) * 2;
            *reinterpret_cast<uint4v*>(dst) = uint4v{w[0], w[1], w[2], w[3]};
            *reinterpret_cast<uint4v*>(dst + 16) = uint4v{w[4], w[5], w[6], w[7]};
        }
    };

    if (tile < num_tiles) stage(0);
    if constexpr (LONG) {
        // one barrier a tile: behind it the tile's product, the staging of the next and the stores of the one before go side by
        // side; one half of the wavefronts begins with the product, the other with the staging
        const bool product_first = wave < C::WAVES / 2;
        if (tile + gridDim.x < num_tiles) issue_loads(tile + gridDim.x);
        __syncthreads();
        for (int it = 0; tile < num_tiles; tile += gridDim.x, ++it) {
            const int cur = it & 1;
            const int64_t next = tile + gridDim.x;
            auto stage_next = [&] {
                if (next < num_tiles) stage(cur ^ 1);
                if (next + gridDim.x < num_tiles) issue_loads(next + gridDim.x);
            };
            if (!product_first) stage_next();
            rotate_tile(xs[cur], os[cur]);
            if (product_first) stage_next();
            if (it > 0) store_tile(tile - gridDim.x, os[cur ^ 1]);
            __syncthreads();
            if (next >= num_tiles) store_tile(tile, os[cur]);
        }
        return;
    }
    __syncthreads();
    for (int it = 0; tile < num_tiles; tile += gridDim.x, ++it) {
        const int cur = it & 1;
        const int64_t next = tile + gridDim.x;
        if (next < num_tiles) issue_loads(next);
        rotate_tile(xs[cur], os[0]);
        __syncthreads();                       // the rotated rows of this tile are complete
        store_tile(tile, os[0]);
        if (next < num_tiles) stage(cur ^ 1);
        __syncthreads();                       // the next tile is staged; `os` is free again
    }
}

template <int D, int DT, bool CACHE, bool LONG>
int launch_decompress_rotate_as(const DecRotSource& src, const float* centroids, const float* rotation, int col_major,
                                void* out, void* out_v, int64_t M, int64_t cap, hipStream_t s) {
    using C = DecRotCfg<D, LONG>;
    const int64_t tiles = (M + C::TT - 1) / C::TT * (CACHE ? 2 : 1);
    hipLaunchKernelGGL((tq4_decompress_rotate_kernel<D, DT, CACHE, LONG>), dim3(unsigned(tiles < cap ? tiles : cap)), dim3(C::THREADS), 0, s,
                       src, centroids, rotation, col_major, static_cast<uint16_t*>(out), static_cast<uint16_t*>(out_v), M, tiles);
    return fq_host::check_launch();
}

template <int D, int DT, bool CACHE>
int launch_decompress_rotate(const DecRotSource& src, const float* centroids, const float* rotation, int col_major,
                             void* out, void* out_v, int64_t M, hipStream_t s) {
    const int64_t cus = fq_host::device_cu_count();
    // At head_dim 256 the matrix in two terms takes 128 registers, and one workgroup of eight wavefronts fills a CU; a second
    // round of workgroups would fetch and split the 256 KB again, so there is one a CU: 2 x 38,400 rows of a cache in bf16
    // 39.2 us with two, 30.2 with one.  Alone on its CU it hides nothing behind another one's work, so from two tiles of 32
    // rows a CU on it is pipelined over tiles of 64 (LONG): 28.0 us; 2 x 192,000 rows 115 in the plain form, 111 pipelined over
    // 32, 108 over 64 (bound by the product: 80 us at the power limit).  2 x 1920 rows 11.9, 12.1 and 13.0.
    if constexpr (D == 256) {
        return M * (CACHE ? 2 : 1) >= 64 * cus
                   ? launch_decompress_rotate_as<D, DT, CACHE, true>(src, centroids, rotation, col_major, out, out_v, M, cus, s)
                   : launch_decompress_rotate_as<D, DT, CACHE, false>(src, centroids, rotation, col_major, out, out_v, M, cus, s);
    } else {
        // workgroups per CU: three fit the LDS; the fp16 route holds two accumulators per wavefront and runs faster with two.
        // (Pipelined, with the second area for rotated rows only two would fit: 2 x 192,128 rows of 128 in bf16 38.8 and 45.3 us.)
        return launch_decompress_rotate_as<D, DT, CACHE, false>(src, centroids, rotation, col_major, out, out_v, M,
                                                                cus * (DT == FQ_F16 ? 2 : 3), s);
    }
}

template <bool CACHE>
int decompress_rotate_any(const DecRotSource& src, const float* centroids, const float* rotation, int col_major, void* out,
                          void* out_v, int dtype, int64_t M, int D, hipStream_t s) {
#define FQ_DECROT_CASE(DD)                                                                                              \
    case DD:                                                                                                            \
        return dtype == FQ_F16                                                                                          \
                   ? launch_decompress_rotate<DD, FQ_F16, CACHE>(src, centroids, rotation, col_major, out, out_v, M, s) \
                   : launch_decompress_rotate<DD, FQ_BF16, CACHE>(src, centroids, rotation, col_major, out, out_v, M, s);
    switch (D) {
        FQ_DECROT_CASE(64)
        FQ_DECROT_CASE(128)
        FQ_DECROT_CASE(256)
        default: return FQ_ERR_UNSUPPORTED_DIM;
    }
#undef FQ_DECROT_CASE
}

}  // namespace
}  // namespace fq

extern "C" int fq_tq4_decompress_rotated(const uint8_t* packed, const float* norms, const float* centroids,
                                         const float* rotation, int rotation_col_major, void* out, int out_dtype,
                                         int64_t M, int D, void* stream) {
    using namespace fq;
    if (M < 0) return FQ_ERR_BAD_SHAPE;
    if (!fq_host::supported_dim(D)) return FQ_ERR_UNSUPPORTED_DIM;
    if (out_dtype != FQ_F16 && out_dtype != FQ_BF16) return FQ_ERR_UNSUPPORTED_DTYPE;
    if (M == 0) return FQ_OK;
    if (!packed || !norms || !centroids || !rotation || !out) return FQ_ERR_NULL_POINTER;
    if (!fq_host::aligned(packed, 4) || !fq_host::aligned(norms, 4) || !fq_host::aligned(rotation, 4) ||
        !fq_host::aligned(out, 16))
        return FQ_ERR_MISALIGNED;
    const DecRotSource src{packed, norms, 1, 1.0f};
    return decompress_rotate_any<false>(src, centroids, rotation, rotation_col_major, out, nullptr, out_dtype, M, D,
                                        static_cast<hipStream_t>(stream));
}

namespace fq_host {
// The keys and values of `tokens` cache rows, rotated back (fq_tq4_decompress_cache has checked the arguments).
int decompress_cache_rotated(const uint8_t* cache, int64_t tokens, int H, int D, const float* centroids,
                             const float* rotation, int col_major, void* out_k, void* out_v, int dtype, void* stream) {
    const fq::DecRotSource src{cache, nullptr, H, 1.0f / float(H)};
    return fq::decompress_rotate_any<true>(src, centroids, rotation, col_major, out_k, out_v, dtype, tokens * H, D,
                                           static_cast<hipStream_t>(stream));
}
}  // namespace fq_host
