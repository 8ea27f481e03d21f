// Block quantize along rows (bi8_quantize_rowwise): per (row, K-block) absmax -> fp32 scale, int8 codes
// rint_even(127 * (x / absmax)).  HBM-bound: every input byte is read once with 128-bit loads, every
// code written once; with two or four rows per wave the scales go through LDS so that each K-block's scales leave the workgroup as
// runs of 8 or 16 consecutive rows (the scale array is block-major / row-minor).
//
// Replaces _quantize_block_rowwise, triton_functions.py:193-216 (one program per row, serial over the
// row's blocks) with a 2-D tiling: one workgroup = 4, 8 or 16 rows x 1 KiB of row, one lane = 16 input bytes,
// one K-block = L adjacent lanes (L = block * sizeof(elem) / 16), absmax by DPP inside the lane group.
#include "bi8_common.h"
#include "bi8_internal.h"

namespace {

constexpr int kThreads = 256;
// Codes leave with ordinary stores.  Marked non-temporal the quantizer by itself is 3-8 % faster, but its codes come back slower to the
// kernel that reads them next.  us, ordinary / non-temporal, the quantizer and quantize + dequantize: bf16, block 128 512 x 4096 3.2 / 2.9, 5.7 /
// 5.6, 3000 x 4096 8.9 / 8.4, 15.7 / 15.8, 8192 x 4096 18.9 / 18.2, 34.9 / 36.6; fp32 1400 x 4096 7.3 / 7.1, 12.7 / 13.1, 8192 x 4096 27.0 / 26.6, 51.8 /
// 55.9; quantize + GEMM bf16 8192 x 11008 -> 1024 148 / 158, fp32 4096 x 12288 -> 4096 252 / 271, 8192 x 4224 -> 2048 95.4 / 95.2.

// One wave = RPW rows x 1 KiB, one workgroup = four of them, one below the other.
// ALIGNED: rows of x on 16-byte boundaries, K a multiple of the elements per 16 bytes, rows of q aligned to their
// 4- or 8-byte stores.  Otherwise (odd row length or leading dimension, e.g. the GPT-2 vocabulary 50257) whole chunks
// move with unaligned 16-byte loads and 4- or 8-byte stores, the last, partial chunk of a row element by element.
// Kp: columns written, K or more: zero codes and zero scales past the row's end (the padding that a GEMM contracted over K wants).
// A row past the end reads the last one and is not stored: the rows' loads do not branch, nor does their arithmetic, so that the rows'
// chains of dependent instructions run side by side: a block that needs the IEEE division (a subnormal, huge or infinite scale, a NaN)
// is done over in one place behind them.
template <int DT, int L, bool ALIGNED, int RPW>
__global__ __launch_bounds__(kThreads) void quantize_rows_vec(const void *__restrict__ x, int8_t *__restrict__ q,
                                                              float *__restrict__ scales, int64_t M, int64_t K, int64_t Kp,
                                                              int64_t ldx, int64_t ldq, int64_t nblk) {
    constexpr int VEC = Bi8Vec<DT>::kElems;
    constexpr int B = L * VEC;                       // block size in elements
    constexpr int TE = BI8_WAVE * VEC;               // elements of one row covered by a tile
    constexpr int NCORR = (DT == BI8_F32) ? 2 : 1;
    constexpr int64_t ES = 16 / VEC;                 // bytes per element

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row0 = (((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * 4 + wave) * RPW;
    if (RPW == 1 && row0 >= M) return;
    const int64_t col0 = (int64_t)blockIdx.x * TE;
    const int64_t left = K - col0;                   // elements of a row from the tile's first column on (none or less: padding only)
    const char *xb = (const char *)x + col0 * ES;

    auto row_of = [&](int i) { return row0 + i < M ? row0 + i : M - 1; };
    const int mine = (int)(left < TE ? (left > 0 ? left : 0) : TE) - lane * VEC;      // of the row's elements from this lane's first on

    bi8_v4u raw[RPW];
#pragma unroll
    for (int i = 0; i < RPW; ++i) raw[i] = bi8_v4u{0u, 0u, 0u, 0u};
    if (mine >= VEC) {
#pragma unroll
        for (int i = 0; i < RPW; ++i) {
            const char *src = xb + row_of(i) * ldx * ES;
            if constexpr (ALIGNED) raw[i] = __builtin_nontemporal_load((const bi8_v4u *)(src + lane * 16));
            else raw[i] = *(const bi8_v4u_unaligned *)(src + lane * 16);
        }
    }
    if constexpr (!ALIGNED) {
        if (mine > 0 && mine < VEC) {                // the row ends inside this chunk
#pragma unroll
            for (int i = 0; i < RPW; ++i) {
                const char *src = xb + row_of(i) * ldx * ES + lane * 16;
#pragma unroll
                for (int e = 0; e < VEC - 1; ++e) {
                    if (e < mine) {
                        if constexpr (DT == BI8_F32) raw[i][e] = ((const uint32_t *)src)[e];
                        else raw[i][e >> 1] |= (uint32_t)((const uint16_t *)src)[e] << (16 * (e & 1));
                    }
                }
            }
        }
    }

    float m[RPW];
    uint32_t w[RPW][VEC / 4];
    bool slow = false;
#pragma unroll
    for (int i = 0; i < RPW; ++i) m[i] = bi8_magnitude_of<DT>(bi8_group_bits<DT, L>(bi8_magnitude_bits<DT>(raw[i])));
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
        float f[VEC];
        bi8_unpack<DT>(raw[i], f);
        slow |= !bi8_scale_is_fast(m[i]);
        const float y = bi8_recip_of_scale(m[i]);
        uint32_t code[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) code[e] = bi8_code_fast<NCORR>(f[e], m[i], y);
#pragma unroll
        for (int e = 0; e < VEC; e += 4) w[i][e / 4] = bi8_pack4(code[e], code[e + 1], code[e + 2], code[e + 3]);
    }
    if (__builtin_expect(__any(slow), 0)) {
#pragma unroll
        for (int i = 0; i < RPW; ++i) {
            if (!bi8_scale_is_fast(m[i])) {                             // (the same for all lanes of a block)
                float f[VEC], s = 0.0f;
                bi8_unpack<DT>(raw[i], f);
#pragma unroll
                for (int e = 0; e < VEC; ++e) s = __builtin_fmaxf(s, __builtin_fabsf(f[e]));      // ignores NaN
                s = bi8_group_max<L>(s);
                m[i] = s;
                uint32_t code[VEC];
#pragma unroll
                for (int e = 0; e < VEC; ++e) code[e] = bi8_code_slow(f[e], s);
#pragma unroll
                for (int e = 0; e < VEC; e += 4) w[i][e / 4] = bi8_pack4(code[e], code[e + 1], code[e + 2], code[e + 3]);
            }
        }
    }

    const int64_t to_write = Kp - col0;
    const int room = (int)(to_write < TE ? to_write : TE) - lane * VEC;          // columns to write from this lane's first on
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
        if (row0 + i >= M) break;
        int8_t *dst = q + (row0 + i) * ldq + col0 + lane * VEC;
        if (room >= VEC) {
            if constexpr (VEC == 4) {
                if constexpr (ALIGNED) *(uint32_t *)dst = w[i][0];
                else *(bi8_u32_unaligned *)dst = w[i][0];
            } else {
                const bi8_v2u c = {w[i][0], w[i][1]};
                if constexpr (ALIGNED) *(bi8_v2u *)dst = c;
                else *(bi8_v2u_unaligned *)dst = c;
            }
        } else if constexpr (!ALIGNED) {
#pragma unroll
            for (int e = 0; e < VEC - 1; ++e)
                if (e < room) dst[e] = (int8_t)((w[i][e / 4] >> (8 * (e & 3))) & 0xffu);
        }
    }
    // The scales: straight from the lanes that hold them, or through LDS, so that each block's leave as a run of all the workgroup's rows.
    const int64_t jb0 = col0 / B;
    if constexpr (RPW == 1) {
        const int64_t jb = jb0 + lane / L;
        if ((lane & (L - 1)) == 0 && jb < nblk) scales[jb * M + row0] = m[0];
    } else {
        constexpr int kRows = 4 * RPW, NB = BI8_WAVE / L;
        __shared__ float s_tile[NB][kRows + 1];
        if ((lane & (L - 1)) == 0) {
#pragma unroll
            for (int i = 0; i < RPW; ++i) s_tile[lane / L][wave * RPW + i] = m[i];
        }
        __syncthreads();
        const int64_t first = row0 - wave * RPW;
        for (int t = threadIdx.x; t < NB * kRows; t += kThreads) {
            const int j = t / kRows, r = t % kRows;
            if (first + r < M && jb0 + j < nblk) scales[(jb0 + j) * M + first + r] = s_tile[j][r];
        }
    }
}

// Any block size, any alignment: one wave per (row, block); lanes stride over the block.
template <int DT>
__global__ __launch_bounds__(kThreads) void quantize_rows_generic(const void *__restrict__ x, int8_t *__restrict__ q,
                                                                  float *__restrict__ scales, int64_t M, int64_t K,
                                                                  int64_t ldx, int64_t ldq, int64_t nblk, int block) {
    const int lane = threadIdx.x & 63;
    const int64_t wave0 = (int64_t)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
    const int64_t nwaves = (int64_t)gridDim.x * (kThreads / 64);
    const int64_t units = M * nblk;
    for (int64_t u = wave0; u < units; u += nwaves) {       // wave-uniform trip count
        // consecutive waves take consecutive blocks of one row
        const int64_t row = u / nblk, j = u % nblk;
        const int64_t k0 = j * block;
        const int64_t n = (K - k0 < block) ? (K - k0) : block;
        float m = 0.0f;
        for (int64_t k = lane; k < n; k += 64) m = __builtin_fmaxf(m, __builtin_fabsf(bi8_load_elem<DT>(x, row * ldx + k0 + k)));
        m = bi8_group_max<64>(m);
        if (lane == 0) scales[j * M + row] = m;
        for (int64_t k = lane; k < n; k += 64) {
            const float v = bi8_load_elem<DT>(x, row * ldx + k0 + k);
            q[row * ldq + k0 + k] = (int8_t)(bi8_code_slow(v, m) & 0xffu);
        }
    }
}

template <int DT, int L, bool ALIGNED, int RPW>
int launch_rows(const void *x, int8_t *q, float *scales, int64_t M, int64_t K, int64_t Kp, int64_t ldx, int64_t ldq, hipStream_t st) {
    constexpr int VEC = Bi8Vec<DT>::kElems;
    constexpr int B = L * VEC;
    constexpr int TE = BI8_WAVE * VEC;
    constexpr int64_t kGridY = 32768;
    const int64_t tiles_k = (Kp + TE - 1) / TE, tiles_m = (M + 4 * RPW - 1) / (4 * RPW);
    const int64_t gy = tiles_m < kGridY ? tiles_m : kGridY, gz = (tiles_m + gy - 1) / gy;
    if (tiles_k * gy * gz > 0x7fffffffLL || gz > 65535) return BI8_ERR_TOO_LARGE;
    const int64_t nblk = (Kp + B - 1) / B;
    hipLaunchKernelGGL((quantize_rows_vec<DT, L, ALIGNED, RPW>), dim3((unsigned)tiles_k, (unsigned)gy, (unsigned)gz), dim3(kThreads), 0, st, x, q, scales, M, K, Kp,
                       ldx, ldq, nblk);
    return bi8_launch_rc();
}
// Rows per wave: one where that leaves every CU at most 24 waves (a call of few rows is latency, and a wave's rows follow one another),
// two up to 72, four beyond, where more loads in flight per wave pay.  us with 1 / 2 / 4 (before: four, 1 KiB loads that waited for
// one another, and the IEEE path inside each row): bf16, block 128 16 x 4096 1.8 / 2.1 / 2.5 (2.8), 512 x 4096 2.6 / 2.7 / 2.9 (3.2), 2048 x
// 4096 7.2 / 6.6 / 6.9 (7.4), 3000 x 4096 9.4 / 9.0 / 8.8 (9.3), 4096 x 4096 11.9 / 11.5 / 10.8 (11.5), 8192 x 8192 37.2 / 34.8 / 35.3 (35.4);
// fp16 100 x 11008 2.3 / 2.7 / 3.0 (3.9), 300 x 16384 4.9 / 4.8 / 5.3 (5.4); fp32, block 32 1000 x 5004 7.6 / 7.5 / 7.0 (7.2).
// Rows off 16-byte boundaries run with one whatever the size where a KiB of row holds at most eight blocks: bf16, block 128 1000 x 5003
// 5.6 / 5.6 / 7.2 (9.1), 8192 x 50257 250 / 279 / 280 (278), block 64 267 / 290 / 287 (282); fp32, block 32 8192 x 50257 472 / 514 / 516 (505).
// With one row per wave every scale is a 4-byte store by itself; smaller blocks, sixteen stores and more per KiB, go with two rows in
// larger calls: from the line for aligned rows on, L = 4 from the next, where codes in the caches are read behind it (quantize + dequantize,
// bf16 block 32 2000 x 3001 12.0 with one, 13.5 with two; 2000 x 5003 17.2 / 16.7), and there not where a row of 16-bit elements is two to four
// runs; with four only at L = 1.  us with 1 / 2 / 4, from memory: bf16, block 32 4810 x 3658 16.0 / 14.7 / 15.1 (with 4 before: 19.0), 6000 x 5003 25.2 /
// 23.2 / 24.0, 8192 x 50257 320 / 317 / 297, 8192 x 2001 15.0 / 15.2 / 15.2; fp16, block 32 2000 x 5003 10.6 / 10.0 / 11.3 (13.0), 4810 x 3658 15.9 / 15.1 /
// 17.6, 8192 x 2001 14.9 / 16.3 / 17.6, 20000 x 1001 17.9 / 19.8 / 21.6, 65536 x 251 28.7 / 25.5 / 29.0 (28.3); bf16, block 16 2000 x 5003 12.3 / 10.2 / 10.7, 8192 x
// 2001 17.4 / 15.6 / 15.6; block 8 8192 x 50257 672 / 473 / 352 (343), 8192 x 5001 53.4 / 40.6 / 34.3 (35.9); fp32, block 16 4000 x 3001 16.8 / 15.3 / 15.4.
constexpr int64_t kOneRowWaves = 24 * 256, kTwoRowWaves = 72 * 256;
template <int DT, int L, bool ALIGNED>
int launch_vec(const void *x, int8_t *q, float *scales, int64_t M, int64_t K, int64_t Kp, int64_t ldx, int64_t ldq, hipStream_t st) {
    constexpr int TE = BI8_WAVE * Bi8Vec<DT>::kElems;
    const int64_t runs = (Kp + TE - 1) / TE, waves = M * runs;
    if constexpr (ALIGNED || L == 1) {
        if (waves > kTwoRowWaves && (ALIGNED || runs > 4)) return launch_rows<DT, L, ALIGNED, 4>(x, q, scales, M, K, Kp, ldx, ldq, st);
        if (waves > kOneRowWaves) return launch_rows<DT, L, ALIGNED, 2>(x, q, scales, M, K, Kp, ldx, ldq, st);
    } else if constexpr (L == 2 || L == 4) {
        if (waves > (L == 4 ? kTwoRowWaves : kOneRowWaves) && (L == 2 || DT == BI8_F32 || runs > 4 || runs == 1))
            return launch_rows<DT, L, ALIGNED, 2>(x, q, scales, M, K, Kp, ldx, ldq, st);
    }
    return launch_rows<DT, L, ALIGNED, 1>(x, q, scales, M, K, Kp, ldx, ldq, st);
}

template <int DT, bool ALIGNED>
int dispatch_vec(const void *x, int8_t *q, float *scales, int64_t M, int64_t K, int64_t Kp, int64_t ldx, int64_t ldq, int lanes, hipStream_t st) {
    switch (lanes) {
    case 1: return launch_vec<DT, 1, ALIGNED>(x, q, scales, M, K, Kp, ldx, ldq, st);
    case 2: return launch_vec<DT, 2, ALIGNED>(x, q, scales, M, K, Kp, ldx, ldq, st);
    case 4: return launch_vec<DT, 4, ALIGNED>(x, q, scales, M, K, Kp, ldx, ldq, st);
    case 8: return launch_vec<DT, 8, ALIGNED>(x, q, scales, M, K, Kp, ldx, ldq, st);
    case 16: return launch_vec<DT, 16, ALIGNED>(x, q, scales, M, K, Kp, ldx, ldq, st);
    case 32: return launch_vec<DT, 32, ALIGNED>(x, q, scales, M, K, Kp, ldx, ldq, st);
    default: return launch_vec<DT, 64, ALIGNED>(x, q, scales, M, K, Kp, ldx, ldq, st);
    }
}

template <int DT>
int dispatch(const void *x, int8_t *q, float *scales, int64_t M, int64_t K, int64_t Kp, int64_t ldx, int64_t ldq, int block, hipStream_t st) {
    constexpr int VEC = Bi8Vec<DT>::kElems;
    // one K-block = 1 .. 64 lanes of 16 input bytes each
    const bool vec_ok = bi8_pow2(block) && block >= VEC && block <= 64 * VEC && bi8_aligned(x, 16 / VEC);
    if (vec_ok) {
        const bool aligned = K % VEC == 0 && Kp % VEC == 0 && ldx % VEC == 0 && ldq % VEC == 0 && bi8_aligned(x, 16) && bi8_aligned(q, VEC);
        return aligned ? dispatch_vec<DT, true>(x, q, scales, M, K, Kp, ldx, ldq, block / VEC, st)
                       : dispatch_vec<DT, false>(x, q, scales, M, K, Kp, ldx, ldq, block / VEC, st);
    }
    if (Kp != K) return BI8_ERR_UNSUPPORTED;
    const int64_t nblk = (K + block - 1) / block;
    const int64_t units = M * nblk;
    int64_t grid = (units + 3) / 4;
    if (grid > 65536) grid = 65536;
    hipLaunchKernelGGL((quantize_rows_generic<DT>), dim3((unsigned)grid), dim3(kThreads), 0, st, x, q, scales, M, K, ldx, ldq, nblk,
                       block);
    return bi8_launch_rc();
}

}  // namespace

extern "C" int bi8x_quantize_rowwise(const void *x, int x_dtype, int8_t *q, float *scales, int64_t M, int64_t K, int64_t Kp, int64_t ldx,
                                     int64_t ldq, int block, void *stream) {
    if (x_dtype < 0 || x_dtype > 2) return BI8_ERR_BAD_DTYPE;
    if (block < 1 || block > (1 << 20)) return BI8_ERR_BAD_BLOCK;
    if (M < 0 || K < 0 || Kp < K || ldx < K || ldq < Kp) return BI8_ERR_BAD_SHAPE;
    if (M == 0 || K == 0) return BI8_OK;
    if (!x || !q || !scales) return BI8_ERR_NULL_POINTER;
    hipStream_t st = (hipStream_t)stream;
    switch (x_dtype) {
    case BI8_F32: return dispatch<BI8_F32>(x, q, scales, M, K, Kp, ldx, ldq, block, st);
    case BI8_BF16: return dispatch<BI8_BF16>(x, q, scales, M, K, Kp, ldx, ldq, block, st);
    default: return dispatch<BI8_F16>(x, q, scales, M, K, Kp, ldx, ldq, block, st);
    }
}

extern "C" int bi8_quantize_rowwise(const void *x, int x_dtype, int8_t *q, float *scales, int64_t M, int64_t K, int64_t ldx,
                                    int64_t ldq, int block, void *stream) {
    return bi8x_quantize_rowwise(x, x_dtype, q, scales, M, K, K, ldx, ldq, block, stream);
}
