// Block dequantize (bi8_dequantize_rowwise): out = (scale * float(code)) * fp32(1/127), cast on store.
// Replaces _dequantize_block_rowwise, triton_functions.py:468-490.  HBM-bound: one lane = one 128-bit store
// of outputs (8 bf16/f16 or 4 fp32) per step, so every wave store covers 1 KiB of contiguous output.  Same
// tiling as the quantizer: a workgroup owns 8 rows x 2 KiB of output row (small calls: 4 x 1 KiB, short rows 8 or 16 x 1 KiB, ragged ones of
// middling calls 4 x 4 KiB) and, with more than a row per wave, first pulls its scales in through LDS, so the block-major / row-minor
// scale array is read as runs of 8 or 16 rows.
#include "bi8_common.h"

namespace {

constexpr int kThreads = 256;

// One lane = kOut outputs = one 16-byte store (8 bf16/f16 or 4 fp32), so every store instruction of a wave
// writes 1 KiB of contiguous output; the codes come in as one 8- or 4-byte load per lane.
template <int DT> struct Out {
    static constexpr int kElems = (DT == BI8_F32) ? 4 : 8;
};

template <int DT, bool ALIGNED> __device__ __forceinline__ void store_vec(void *out, int64_t idx, const float *v) {
    if constexpr (DT == BI8_F32) {
        const bi8_v4u w = {__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
        if constexpr (ALIGNED) __builtin_nontemporal_store(w, (bi8_v4u *)((float *)out + idx));
        else *(bi8_v4u_unaligned *)((float *)out + idx) = w;
    } else {
        bi8_v4u w;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint32_t lo, hi;
            if constexpr (DT == BI8_BF16) {
                lo = bi8_bf16_bits(v[2 * e]);
                hi = bi8_bf16_bits(v[2 * e + 1]);
            } else {
                lo = bi8_f16_bits(v[2 * e]);
                hi = bi8_f16_bits(v[2 * e + 1]);
            }
            w[e] = lo | (hi << 16);
        }
        if constexpr (ALIGNED) __builtin_nontemporal_store(w, (bi8_v4u *)((uint16_t *)out + idx));
        else *(bi8_v4u_unaligned *)((uint16_t *)out + idx) = w;
    }
}

// One wave = R rows x NC chunks of 64 * kOut codes, one workgroup = four of them, one below the other.
// ALIGNED: rows of q on boundaries of their 4- or 8-byte loads, rows of out on 16-byte boundaries, K a multiple of the elements per
// store.  Otherwise (odd row lengths) whole chunks move with unaligned accesses and the last, partial chunk of a row element by
// element, as in the quantizer; these stores are not marked non-temporal: a wave's run starts and ends inside a cache line whose
// other part comes from the next wave, and the two are to meet in the L2.  Quantize + dequantize of fp32 [1000,5003], block 32:
// 19.0 -> 15.3 us against dequantize_rows_generic (one code, one division and one scale read per output).
template <int DT, bool ALIGNED, int R, int NC>
__global__ __launch_bounds__(kThreads) void dequantize_rows_vec(const int8_t *__restrict__ q, const float *__restrict__ scales,
                                                                void *__restrict__ out, int64_t M, int64_t K, int64_t ldq,
                                                                int64_t ldo, int64_t nblk, int log2b) {
    constexpr int VEC = Out<DT>::kElems;
    constexpr int kRows = 4 * R;
    constexpr int TE = NC * BI8_WAVE * VEC;        // codes per tile row
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t first = ((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * kRows, row0 = first + wave * R;
    if (R == 1 && row0 >= M) return;
    const int64_t col0 = (int64_t)blockIdx.x * TE;
    const int64_t jb0 = col0 >> log2b;
    const int left = (int)(K - col0 < TE ? K - col0 : TE);          // of a row's codes, from the tile's first column on
    auto row_of = [&](int i) { return row0 + i < M ? row0 + i : M - 1; };

    uint32_t raw[R][NC][VEC / 4];
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < VEC / 4; ++e) raw[i][c][e] = 0u;
    auto load = [&](int i, int c) {
        const int8_t *src = q + row_of(i) * ldq + col0 + c * BI8_WAVE * VEC + lane * VEC;
        if constexpr (VEC == 8) {
            const bi8_v2u v = ALIGNED ? __builtin_nontemporal_load((const bi8_v2u *)src) : (bi8_v2u)*(const bi8_v2u_unaligned *)src;
            raw[i][c][0] = v[0];
            raw[i][c][1] = v[1];
        } else {
            raw[i][c][0] = ALIGNED ? __builtin_nontemporal_load((const uint32_t *)src) : (uint32_t)*(const bi8_u32_unaligned *)src;
        }
    };
    if (left == TE) {                              // (one branch: the first use of a load need not wait for the others)
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int c = 0; c < NC; ++c) load(i, c);
    } else {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int mine = left - (c * BI8_WAVE + lane) * VEC;          // of the row's codes from this lane's first on
            if (mine >= VEC) {
#pragma unroll
                for (int i = 0; i < R; ++i) load(i, c);
            } else if (!ALIGNED && mine > 0) {                            // the row ends inside this chunk
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    const int8_t *src = q + row_of(i) * ldq + col0 + (c * BI8_WAVE + lane) * VEC;
#pragma unroll
                    for (int e = 0; e < VEC - 1; ++e)
                        if (e < mine) raw[i][c][e >> 2] |= (uint32_t)(uint8_t)src[e] << (8 * (e & 3));
                }
            }
        }
    }

    // one row per wave: its scales straight from memory; otherwise through LDS, read as runs of the workgroup's rows
    constexpr int kMaxBlocks = R == 1 ? 1 : TE / 8;                       // block size >= 8 on this path
    __shared__ float s_tile[kMaxBlocks][kRows + 1];
    float s_lane[NC];
    if constexpr (R == 1) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int incol = (c * BI8_WAVE + lane) * VEC;
            s_lane[c] = incol < left ? scales[(jb0 + (incol >> log2b)) * M + row0] : 0.0f;
        }
    } else {
        const int nb = (TE >> log2b) > 0 ? (TE >> log2b) : 1;             // blocks per tile row
        for (int t = tid; t < nb * kRows; t += kThreads) {
            const int j = t / kRows, r = t % kRows;
            float s = 0.0f;
            if (first + r < M && jb0 + j < nblk) s = scales[(jb0 + j) * M + first + r];
            s_tile[j][r] = s;
        }
        __syncthreads();
    }

    const float inv127 = (float)(1.0 / 127.0);
#pragma unroll
    for (int i = 0; i < R; ++i) {
        if (row0 + i >= M) break;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int incol = (c * BI8_WAVE + lane) * VEC, mine = left - incol;
            if (mine <= 0) continue;
            const float s = R == 1 ? s_lane[c] : s_tile[R == 1 ? 0 : incol >> log2b][wave * R + i];
            float v[VEC];
#pragma unroll
            for (int e = 0; e < VEC / 4; ++e) {
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const int code = (int)(raw[i][c][e] << (24 - 8 * b)) >> 24;     // sign-extended byte b
                    v[4 * e + b] = (s * (float)code) * inv127;                      // two roundings, left to right
                }
            }
            const int64_t at = (row0 + i) * ldo + col0 + incol;
            if (ALIGNED || mine >= VEC) {
                store_vec<DT, ALIGNED>(out, at, v);
            } else {
#pragma unroll
                for (int e = 0; e < VEC - 1; ++e)
                    if (e < mine) bi8_store_elem<DT>(out, at + e, v[e]);
            }
        }
    }
}

template <int DT, bool ALIGNED, int R, int NC>
int launch_rows(const int8_t *q, const float *scales, void *out, int64_t M, int64_t K, int64_t ldq, int64_t ldo, int block, hipStream_t st) {
    constexpr int TE = NC * BI8_WAVE * Out<DT>::kElems;
    constexpr int64_t kGridY = 32768;
    const int64_t tiles_k = (K + TE - 1) / TE, tiles_m = (M + 4 * R - 1) / (4 * R);
    const int64_t gy = tiles_m < kGridY ? tiles_m : kGridY, gz = (tiles_m + gy - 1) / gy;
    if (tiles_k * gy * gz > 0x7fffffffLL || gz > 65535) return BI8_ERR_TOO_LARGE;
    hipLaunchKernelGGL((dequantize_rows_vec<DT, ALIGNED, R, NC>), dim3((unsigned)tiles_k, (unsigned)gy, (unsigned)gz), dim3(kThreads), 0, st, q, scales, out, M, K, ldq, ldo,
                       (K + block - 1) / block, __builtin_ctz((unsigned)block));
    return bi8_launch_rc();
}

template <int DT>
__global__ __launch_bounds__(kThreads) void dequantize_rows_generic(const int8_t *__restrict__ q, const float *__restrict__ scales,
                                                                    void *__restrict__ out, int64_t M, int64_t K, int64_t ldq,
                                                                    int64_t ldo, int block) {
    // one workgroup per (row, run of 2048 columns): consecutive lanes take consecutive elements, no 64-bit division
    const float inv127 = (float)(1.0 / 127.0);
    const int64_t runs = (K + 2047) / 2048;
    const int64_t units = M * runs;
    for (int64_t u = blockIdx.x; u < units; u += gridDim.x) {
        const int64_t row = u / runs, k0 = (u % runs) * 2048;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int64_t k = k0 + t * kThreads + threadIdx.x;
            if (k < K) {
                const float s = scales[(k / block) * M + row];
                bi8_store_elem<DT>(out, row * ldo + k, (s * (float)q[row * ldq + k]) * inv127);
            }
        }
    }
}

// One row and one chunk per wave where that is few waves (a call of few rows is latency), else two rows of two chunks.  us with one / two
// rows (before: two, loads that waited for one another), codes in the caches: bf16, block 128 16 x 4096 1.7 / 2.4 (2.7), 512 x 4096 2.6 /
// 3.1 (3.2), 2048 x 4096 6.3 / 5.2 (5.1), 8192 x 8192 37.3 / 32.6 (33.6); fp16 100 x 11008 2.1 / 2.8 (2.9), 300 x 16384 4.3 / 3.9 (4.1).
// Rows of one chunk: two or four of them.  Codes from memory, block 32, one / two / four: bf16 12000 x 256 4.8 / 3.6 / 3.8 (3.6), 24000 x 256 7.4 /
// 6.0 / 5.4 (6.0), 65536 x 256 17.4 / 13.6 / 12.7 (13.6), 24000 x 512 9.9 / 9.0 / 7.6 (9.0), 36000 x 512 13.9 / 12.6 / 13.0 (12.6); fp32 12000 x 256 4.9 / 3.8 /
// 3.8 (4.0), 24000 x 256 8.9 / 7.2 / 6.0 (7.2), 65536 x 256 21.0 / 16.5 / 17.4 (16.6).  Off 16-byte boundaries one or four: bf16 12000 x 251 6.2 for one, 7.2
// for four (6.2), 65536 x 251 31.2 / 25.6 (26.5), fp32 33.0 / 28.6 (28.0).
// Rows off 16-byte boundaries: one chunk per wave in larger calls too (fp32 larger than 16-bit ones), then one row of four chunks (a wave's run
// cuts lines at its two ends only) where these fill five of six waves' chunks at least and a chunk holds few scales (blocks from 32 on: a wave
// of one row reads each from memory by itself).  Codes from memory, 1 x 1, 1 x 4, 2 x 2 (before: 2 x 2, loads that waited for one another): bf16
// block 32 1500 x 5003 8.9, 8.4, 9.3 (9.3), 1900 x 5003 10.9, 9.9, 10.6 (10.5), 2600 x 5003 14.3, 13.3, 13.9 (13.8), 1300 x 10001 13.7, 13.0, 12.4 (12.1); block 128
// 2300 x 5003 13.5, 11.5, 13.0 (12.4); fp32 block 32 1200 x 5003 11.4, 9.9, 10.2 (10.3), 900 x 10001 14.0, 12.8, 12.9 (13.0), 6000 x 5003 block 16 43, 42, 37 (40).  Filled less: bf16
// block 32 4500 x 2049 10.1, 12.9, 8.9 (9.0), 2500 x 3001 8.0, 7.9, 8.6 (8.7), 4000 x 3001 13.1, 14.2, 12.5 (11.6), fp32 4000 x 1201 8.5, 8.3, 7.3 (7.4).  More scales: bf16 block 16
// 1500 x 5003 9.1, 9.5, 10.0 (9.9), 3000 x 3001 10.3, 11.7, 9.9 (9.8), fp32 3000 x 3001 14.3, 15.0, 14.0 (13.7).
constexpr int64_t kOneRunWaves = 24 * 256, kOneShortRowWavesRagged = 96 * 256;
template <int DT> constexpr int64_t kOneRunWavesRagged = (DT == BI8_F32 ? 88 : 64) * 256;
template <int DT> constexpr int64_t kOneRunWavesFilled = (DT == BI8_F32 ? 88 : 56) * 256;
template <int DT> constexpr int64_t kOneRowWavesFilled = (DT == BI8_F32 ? 144 : 96) * 256;
constexpr int64_t kTwoShortRowsWaves = 64 * 256, kFourLongerRowsWaves = 128 * 256;
template <int DT, bool ALIGNED>
int launch_vec(const int8_t *q, const float *scales, void *out, int64_t M, int64_t K, int64_t ldq, int64_t ldo, int block, hipStream_t st) {
    constexpr int kChunk = BI8_WAVE * Out<DT>::kElems;
    const int64_t runs = (K + kChunk - 1) / kChunk, waves = M * runs;
    const bool filled = !ALIGNED && block >= 32 && 6 * runs >= 5 * 4 * ((runs + 3) / 4);      // ... with waves of one row of four chunks
    if (waves <= (ALIGNED ? kOneRunWaves : K <= kChunk ? kOneShortRowWavesRagged : filled ? kOneRunWavesFilled<DT> : kOneRunWavesRagged<DT>))
        return launch_rows<DT, ALIGNED, 1, 1>(q, scales, out, M, K, ldq, ldo, block, st);
    if (K <= kChunk) {
        if constexpr (ALIGNED)
            if (waves <= kTwoShortRowsWaves || (2 * K > kChunk && waves > kFourLongerRowsWaves)) return launch_rows<DT, ALIGNED, 2, 1>(q, scales, out, M, K, ldq, ldo, block, st);
        return launch_rows<DT, ALIGNED, 4, 1>(q, scales, out, M, K, ldq, ldo, block, st);
    }
    if constexpr (!ALIGNED)
        if (filled && waves <= kOneRowWavesFilled<DT>) return launch_rows<DT, ALIGNED, 1, 4>(q, scales, out, M, K, ldq, ldo, block, st);
    return launch_rows<DT, ALIGNED, 2, 2>(q, scales, out, M, K, ldq, ldo, block, st);
}

template <int DT>
int dispatch(const int8_t *q, const float *scales, void *out, int64_t M, int64_t K, int64_t ldq, int64_t ldo, int block,
             hipStream_t st) {
    constexpr int VEC = Out<DT>::kElems;
    // Blocks that no chunk straddles, and elements on boundaries of their own size (what the unaligned accesses need); a row shorter
    // than a chunk would be all element by element.
    const bool vec_ok = bi8_pow2(block) && block >= 8 && K >= VEC && bi8_aligned(out, DT == BI8_F32 ? 4 : 2);
    if (vec_ok) {
        const bool aligned = K % VEC == 0 && ldq % VEC == 0 && ldo % VEC == 0 && bi8_aligned(q, VEC) && bi8_aligned(out, 16);
        return aligned ? launch_vec<DT, true>(q, scales, out, M, K, ldq, ldo, block, st) : launch_vec<DT, false>(q, scales, out, M, K, ldq, ldo, block, st);
    }
    int64_t grid = M * ((K + 2047) / 2048);
    if (grid > (1 << 20)) grid = 1 << 20;
    hipLaunchKernelGGL((dequantize_rows_generic<DT>), dim3((unsigned)grid), dim3(kThreads), 0, st, q, scales, out, M, K, ldq, ldo,
                       block);
    return bi8_launch_rc();
}

}  // namespace

extern "C" int bi8_dequantize_rowwise(const int8_t *q, const float *scales, void *out, int out_dtype, int64_t M, int64_t K,
                                      int64_t ldq, int64_t ldo, int block, void *stream) {
    if (out_dtype < 0 || out_dtype > 2) return BI8_ERR_BAD_DTYPE;
    if (block < 1 || block > (1 << 20)) return BI8_ERR_BAD_BLOCK;
    if (M < 0 || K < 0 || ldq < K || ldo < K) return BI8_ERR_BAD_SHAPE;
    if (M == 0 || K == 0) return BI8_OK;
    if (!q || !scales || !out) return BI8_ERR_NULL_POINTER;
    hipStream_t st = (hipStream_t)stream;
    switch (out_dtype) {
    case BI8_F32: return dispatch<BI8_F32>(q, scales, out, M, K, ldq, ldo, block, st);
    case BI8_BF16: return dispatch<BI8_BF16>(q, scales, out, M, K, ldq, ldo, block, st);
    default: return dispatch<BI8_F16>(q, scales, out, M, K, ldq, ldo, block, st);
    }
}
