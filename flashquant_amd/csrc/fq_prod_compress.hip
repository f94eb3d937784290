// TurboQuantProd key compress for gfx950: 3-bit Lloyd-Max index + 1 sign bit of the
// sketched residual per coordinate, packed as one nibble (sign << 3 | index), plus the
// row norm and the residual norm.
//
// Operator: TurboQuantProd.quantize (src/flashquant/core/quantizer.py:285-304):
//   n = ||x||, y = (x / (n + 1e-10)) R^T, idx = #{boundaries < y}        (the bits-1 codebook)
//   resid = x - (centroids[idx] R) n,  gamma = ||resid||,  signs = sign(resid S^T), 0 -> +1
// The residual is handled in rotated space: resid R^T = (n + 1e-10) y - n centroids[idx]
// has the same norm (R is orthogonal) and resid S^T = (resid R^T) (S R^T)^T, so the second
// product uses the matrix W = S R^T, which the caller computes once.
//
// Both products run on the float32 MFMA (v_mfma_f32_16x16x4_f32): the signs of small
// projections are decided at float32 accuracy, as in the reference.  A workgroup of 4
// wavefronts takes 16 rows at a time; wavefront w owns output columns 16w..16w+15 and
// 64+16w.. of both products and keeps those columns of R and W in registers for the
// kernel's lifetime.
#include "fq_common.hpp"
#include "fq_device.hpp"

namespace fq {

constexpr int kPcRows = 16;
constexpr int kPcStride = 128 + 4;   // floats per staged row

template <int DT>
__global__ __launch_bounds__(256) void prod_compress_kernel(
    const uint4v* __restrict__ x, const float* __restrict__ R, int rot_col_major, const float* __restrict__ W,
    const float* __restrict__ boundaries, const float* __restrict__ centroids, uint32_t* __restrict__ packed,
    float* __restrict__ norms, float* __restrict__ gamma, int64_t M, int64_t num_tiles) {
    constexpr int D = 128;
    __shared__ float xs[kPcRows][kPcStride];   // normalised row, then the rotated residual
    __shared__ float ys[kPcRows][kPcStride];   // rotated row, then the projected residual
    __shared__ float bnd[8], cen[8];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int n16 = lane & 15, g4 = lane >> 4;
    const int row = tid >> 4, c8 = tid & 15;   // elementwise phases: 8 coordinates of one row

    if (tid < 7) bnd[tid] = boundaries[tid];
    if (tid == 7) bnd[7] = __builtin_inff();
    if (tid >= 8 && tid < 16) cen[tid - 8] = centroids[tid - 8];

    float rb[2][4][8], wb[2][4][8];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        load_rotation_any<D>(R, rot_col_major != 0, true, 16 * (wave + 4 * i), n16, g4, rb[i]);
        load_rotation_any<D>(W, false, true, 16 * (wave + 4 * i), n16, g4, wb[i]);
    }
    __syncthreads();

    for (int64_t tile = blockIdx.x; tile < num_tiles; tile += gridDim.x) {
        const int64_t grow = tile * kPcRows + row;
        const bool live = grow < M;
        // ---- norm, normalised row --------------------------------------------------------
        float e[8];
        {
            const uint4v raw = live ? x[grow * (D / 8) + c8] : uint4v{0, 0, 0, 0};
            const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                e[2 * i] = load_elem<DT>(uint16_t(w[i] & 0xffffu));
                e[2 * i + 1] = load_elem<DT>(uint16_t(w[i] >> 16));
            }
        }
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) ss = __builtin_fmaf(e[i], e[i], ss);
#pragma unroll
        for (int m = 1; m < 16; m <<= 1) ss += xor_shuffle(ss, m);
        const float nrm = __builtin_sqrtf(ss);
        const float den = nrm + 1e-10f;
#pragma unroll
        for (int i = 0; i < 8; ++i) xs[row][8 * c8 + i] = e[i] / den;
        __syncthreads();

        // ---- y = xhat R^T ------------------------------------------------------------------
        float a[4][8];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int k = 0; k < 8; ++k) a[j][k] = xs[n16][32 * j + 8 * g4 + k];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float4v acc = rotate_block<D>(a, rb[i]);
#pragma unroll
            for (int r = 0; r < 4; ++r) ys[4 * g4 + r][16 * (wave + 4 * i) + n16] = acc[r];
        }
        __syncthreads();

        // ---- 3-bit index, rotated residual, its norm ---------------------------------------------
        uint32_t nib = 0;
        float g2 = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float y = ys[row][8 * c8 + i];
            uint32_t idx = 0;
#pragma unroll
            for (int b = 0; b < 7; ++b) idx += (bnd[b] < y) ? 1u : 0u;
            const float r = den * y - nrm * cen[idx];
            g2 = __builtin_fmaf(r, r, g2);
            xs[row][8 * c8 + i] = r;
            nib |= idx << (4 * i);
        }
#pragma unroll
        for (int m = 1; m < 16; m <<= 1) g2 += xor_shuffle(g2, m);
        __syncthreads();

        // ---- projection of the residual: (resid R^T) W^T ---------------------------------------------
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int k = 0; k < 8; ++k) a[j][k] = xs[n16][32 * j + 8 * g4 + k];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float4v acc = rotate_block<D>(a, wb[i]);
#pragma unroll
            for (int r = 0; r < 4; ++r) ys[4 * g4 + r][16 * (wave + 4 * i) + n16] = acc[r];
        }
        __syncthreads();

        // ---- sign bits, pack: byte j = nibble(2j) << 4 | nibble(2j + 1) ------------------------------------
        uint32_t word = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t neg = ys[row][8 * c8 + i] < 0.0f ? 8u : 0u;
            const uint32_t nb = ((nib >> (4 * i)) & 7u) | neg;
            word |= nb << (8 * (i >> 1) + ((i & 1) ? 0 : 4));
        }
        if (live) {
            packed[grow * (D / 8) + c8] = word;
            if (c8 == 0) {
                norms[grow] = nrm;
                gamma[grow] = __builtin_sqrtf(g2);
            }
        }
        // the next tile's first barrier orders its xs writes after this tile's reads of xs;
        // ys is rewritten only after that barrier as well
    }
}

// One wavefront per token: its row [K nibbles | K norm | K residual norm | V idx | V norm] assembled from the five
// operands and written where its slot says, 4 bytes a lane (W = uint32_t; single bytes where the cache, its row stride
// or an operand is not aligned to 4).  Bound by the launch at a decode step's size and by HBM beyond it.  As torch
// copies into a row buffer and an indexed store it was six launches and twice the bytes: a generated token of 8 sequences
// with its attention 207.7 us, 192.5 with this launch of 5 us.  `kw`, `nw`: units of one index section and of one section of norms.
template <typename W>
__global__ __launch_bounds__(256) void prod_store_rows_kernel(
    W* __restrict__ cache, const int64_t* __restrict__ slots, const W* __restrict__ k_packed, const W* __restrict__ k_norms,
    const W* __restrict__ k_gamma, const W* __restrict__ v_packed, const W* __restrict__ v_norms, int64_t tokens,
    int64_t num_slots, int64_t row_stride, int kw, int nw) {
    const int lane = threadIdx.x & 63;
    const int row_units = 2 * kw + 3 * nw;
    for (int64_t t = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6); t < tokens; t += int64_t(gridDim.x) * 4) {
        int64_t slot = slots[t];
        slot = slot < 0 ? slot + num_slots : slot;   // as an indexed store counts from the end
        if (slot < 0 || slot >= num_slots) continue;
        W* row = cache + slot * row_stride;
        for (int i = lane; i < row_units; i += 64) {
            const W* src;
            int64_t at;
            if (i < kw) { src = k_packed; at = t * kw + i; }
            else if (i < kw + nw) { src = k_norms; at = t * nw + (i - kw); }
            else if (i < kw + 2 * nw) { src = k_gamma; at = t * nw + (i - kw - nw); }
            else if (i < 2 * kw + 2 * nw) { src = v_packed; at = t * kw + (i - kw - 2 * nw); }
            else { src = v_norms; at = t * nw + (i - 2 * kw - 2 * nw); }
            row[i] = src[at];
        }
    }
}

template <typename W>
int launch_prod_store_rows(uint8_t* cache, const int64_t* slots, const uint8_t* kp, const float* kn, const float* kg,
                           const uint8_t* vp, const float* vn, int64_t tokens, int64_t num_slots, int64_t row_stride, int H,
                           int D, unsigned grid, hipStream_t s) {
    constexpr int B = int(sizeof(W));
    auto in = [](const void* p) { return static_cast<const W*>(p); };
    hipLaunchKernelGGL(prod_store_rows_kernel<W>, dim3(grid), dim3(256), 0, s, reinterpret_cast<W*>(cache), slots, in(kp), in(kn),
                       in(kg), in(vp), in(vn), tokens, num_slots, row_stride / B, H * (D / 2) / B, H * 4 / B);
    return fq_host::check_launch();
}

}  // namespace fq

namespace fq_host {
int device_cu_count();
}

extern "C" int fq_prod_store_rows(uint8_t* kv_cache, int64_t row_stride, const int64_t* slot_mapping,
                                  const uint8_t* k_packed, const float* k_norms, const float* k_residual_norms,
                                  const uint8_t* v_packed, const float* v_norms, int64_t num_tokens, int64_t num_slots,
                                  int H, int D, void* stream) {
    using namespace fq;
    if (num_tokens < 0 || num_slots < 0 || H <= 0 || H > 65535 || D <= 0 || D % 2 != 0 || D > 4096) return FQ_ERR_BAD_SHAPE;
    if (row_stride < int64_t(H) * (D + 12)) return FQ_ERR_BAD_SHAPE;
    if (num_tokens == 0) return FQ_OK;
    if (!kv_cache || !slot_mapping || !k_packed || !k_norms || !k_residual_norms || !v_packed || !v_norms)
        return FQ_ERR_NULL_POINTER;
    const int64_t wgs = (num_tokens + 3) / 4, cap = int64_t(fq_host::device_cu_count()) * 8;
    const unsigned grid = unsigned(wgs < cap ? wgs : cap);
    auto launch = [&](auto w) {
        return launch_prod_store_rows<decltype(w)>(kv_cache, slot_mapping, k_packed, k_norms, k_residual_norms, v_packed, v_norms,
                                                   num_tokens, num_slots, row_stride, H, D, grid, static_cast<hipStream_t>(stream));
    };
    const bool words = (H * (D / 2)) % 4 == 0 && row_stride % 4 == 0 && fq_host::aligned(kv_cache, 4) &&
                       fq_host::aligned(k_packed, 4) && fq_host::aligned(v_packed, 4);
    return words ? launch(uint32_t{}) : launch(uint8_t{});
}

extern "C" int fq_prod_compress(const void* x, int x_dtype, const float* rotation, int rotation_col_major,
                                const float* sketch_rot, const float* boundaries, const float* centroids,
                                uint8_t* packed, float* norms, float* residual_norms, int64_t M, int D,
                                void* stream) {
    using namespace fq;
    if (M < 0) return FQ_ERR_BAD_SHAPE;
    if (!fq_host::supported_dim(D) || D != 128) return FQ_ERR_UNSUPPORTED_DIM;
    if (x_dtype != FQ_F16 && x_dtype != FQ_BF16) return FQ_ERR_UNSUPPORTED_DTYPE;
    if (M == 0) return FQ_OK;
    if (!x || !rotation || !sketch_rot || !boundaries || !centroids || !packed || !norms || !residual_norms)
        return FQ_ERR_NULL_POINTER;
    if (!fq_host::aligned(x, 16) || !fq_host::aligned(packed, 4) || !fq_host::aligned(rotation, 16) ||
        !fq_host::aligned(sketch_rot, 16))
        return FQ_ERR_MISALIGNED;
    const int64_t tiles = (M + kPcRows - 1) / kPcRows;
    const int64_t cap = int64_t(fq_host::device_cu_count()) * 4;
    const unsigned grid = unsigned(tiles < cap ? tiles : cap);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const uint4v* xp = static_cast<const uint4v*>(x);
    uint32_t* pp = reinterpret_cast<uint32_t*>(packed);
    if (x_dtype == FQ_F16)
        hipLaunchKernelGGL(prod_compress_kernel<FQ_F16>, dim3(grid), dim3(256), 0, s, xp, rotation, rotation_col_major,
                           sketch_rot, boundaries, centroids, pp, norms, residual_norms, M, tiles);
    else
        hipLaunchKernelGGL(prod_compress_kernel<FQ_BF16>, dim3(grid), dim3(256), 0, s, xp, rotation, rotation_col_major,
                           sketch_rot, boundaries, centroids, pp, norms, residual_norms, M, tiles);
    return fq_host::check_launch();
}
