// Block quantize in both directions at once (bi8_quantize_dual): x [R,C] -> codes [R,C] with scales [ceil(C/B), R]
// (blocks along the rows, what bi8_quantize_rowwise writes) AND codes [C,R] with scales [ceil(R/B), C] (blocks down
// the columns, what bi8_quantize_transposed writes), from one pass over x.  A training step of the reference
// quantizes each of X, W and G twice, once per direction (block_linear.py:77-78, :92-94, :100-103): with this kernel
// every one of them is read from HBM once.
//
// What bounds it: memory, at 4.7 to 5.0 TB/s (58 to 54 us, machine to machine) of the 272 MB of bf16 [8192,8192], block 128 (a copy with
// these access widths: 6.2), behind it ~20
// vector instructions per element.  us, a branch around every load and store, per-element NaN tests and the IEEE path inside each
// row -> this: bf16 block 128 [8192,8192] 57.9 -> 54.2, [4096,11008] 44.4 -> 41.8, [11008,4096] 40.8 -> 39.0; block 64 [8192,3072] with
// column sums 29.0 -> 23.2, [8192,50257] 414 -> 380 ([8192,50304]: 360 -> 345); fp32 [8192,8192] 114 -> 85 (three workgroups per CU for two).
//
// A workgroup owns a 128 x 128 tile, held in registers as two 64-column halves (16 bytes per lane per row pass; the
// next tile's loads are issued while this one is processed).  The row direction is finished straight from the
// registers: the lanes of one row reduce their absmax with DPP, quantize and store their codes.  The column direction
// runs half by half through LDS exactly as in bi8_quantize_transposed (tile kept in its own type, 16-byte LDS accesses).  Both
// outputs are bit for bit those of the two separate entry points.
//
// bi8_quantize_dual_colsum also returns the column sums of x (the bias gradient G.sum(dim=0) of block_linear.py:110,
// when x is the output gradient G): the column walk has every element in a register anyway, so each thread adds up its
// rows, the tile's row groups are added in ascending order, the tiles' sums go to a workspace [tile row][column] and a
// second, tiny kernel adds them in ascending order (fp32 sums in a fixed order: deterministic) and casts.
#include "bi8_common.h"
#include "bi8_internal.h"

namespace {

constexpr int kTR = 128;           // tile rows
constexpr int kTC = 64;            // columns of one half
constexpr int kThreads = 256;
// Tile order, as in bi8_quantize_transposed: the tiles in flight at one time form a compact patch of the matrix
// (bands of kSBR tile rows, chunks of kSBC tile columns inside a band, row by row inside a chunk), so that the reads
// and row-direction writes (runs along the rows) and the column-direction writes (runs down the columns) of the patch
// are all long runs in memory.
// Measured on bf16 [8192,8192]: 16 x 16 tiles 64.0 us, row by row 65.4, 8 x 32 64.6, 32 x 8 69.
constexpr int kSBR = 16, kSBC = 16;
// DOWN: inside a chunk column by column instead of row by row.  Two tiles side by side are then kSBR apart in the order, a multiple of
// the eight XCDs: where rows of x start off 128-byte lines, both read the line that their border cuts, and it is in their L2.
template <bool DOWN> __device__ __forceinline__ void tile_coords(int t, int tiles_r, int tiles_c, int &tr, int &tc) {
    const int band = t / (kSBR * tiles_c);
    const int rows_b = (tiles_r - band * kSBR < kSBR) ? (tiles_r - band * kSBR) : kSBR;
    const int in = t - band * kSBR * tiles_c;
    const int chunk = in / (rows_b * kSBC);
    const int wc = (tiles_c - chunk * kSBC < kSBC) ? (tiles_c - chunk * kSBC) : kSBC;
    const int in2 = in - chunk * rows_b * kSBC;
    tr = band * kSBR + (DOWN ? in2 % rows_b : in2 / wc);
    tc = chunk * kSBC + (DOWN ? in2 / rows_b : in2 % wc);
}
constexpr int kQPitch = kTR + 16;  // code tile pitch in bytes: rows stay 16-byte aligned

// element k (of one or two) of a 32-bit word of x
template <int DT> __device__ __forceinline__ float word_elem(uint32_t d, int k) {
    if constexpr (DT == BI8_F32) return bi8_u2f(d);
    else if constexpr (DT == BI8_BF16) return k == 0 ? bi8_u2f(d << 16) : bi8_u2f(d & 0xffff0000u);
    else return bi8_from_f16_bits(k == 0 ? d & 0xffffu : d >> 16);
}

template <int DT, int B, bool SUM, int NH> struct DualLds {
    static constexpr int kES = DT == BI8_F32 ? 4 : 2;              // bytes per element
    static constexpr int kCPT = 4 / kES;                           // columns per thread in the column walk: one 32-bit word
    static constexpr int kG = kThreads / (kTC / kCPT);             // row groups: 4 (fp32) or 8
    static constexpr int kXPitch = kTC * kES + (kES == 4 ? 0 : 16);      // bytes, 16-byte aligned (as in bi8_quantize_transposed)
    // the tile's row-direction scales, [block along the row][tile row]: stored from here as runs of kTR consecutive rows
    // (single 4-byte stores from the lanes that hold them cost the fabric a 32-byte write each)
    static constexpr int kNRB = (NH * kTC + B - 1) / B;
    __attribute__((aligned(16))) uint8_t x[kTR * kXPitch];
    __attribute__((aligned(16))) uint8_t q[kTC * kQPitch];
    uint32_t max[kG][kTC / kCPT];
    float sum[SUM ? kG : 1][kTC];
    float rs[kNRB][kTR];
};

// ALIGNED: rows of x start on 16-byte boundaries and C is a multiple of the elements per 16 bytes.  Otherwise 16-byte chunks move
// with unaligned accesses, the last, partial chunk of a row as the row's last 16 bytes.
// NH: halves per tile.  2 is the tile described above; 1 (a 128 x 64 tile, blocks of at most 64) doubles the number of
// workgroups for inputs too small to occupy the chip with full tiles.
// Rp, Cp: rows and columns written, the matrix' own or more: zeros past its end.
// FULL: the tiles that lie inside the matrix, otherwise those at its right and lower end.  Every load and store of a full tile is
// unconditional, so that the wait for the next tile's loads is for those, and not for the stores issued behind them: with a branch
// around either the compiler cannot count them and waits for everything, a tile's codes on their way to memory included.  Tiles at the
// ends: a call of few rows is little else, and what bounds it is the chain load, rows, columns, store and the length of the code, run
// once; so no loads element by element, none of rows and passes that lie past the end, loops where single codes are stored.  us,
// with all these -> this (before the two kinds of tiles): block 64 fp32 100 x 11008 7.7 -> 6.0 (6.6), 500 x 4096 8.2 -> 6.6 (7.0), 11008 x 100 9.1 ->
// 6.7 (7.6), bf16 300 x 5003 7.2 -> 6.2 (9.0), 300 x 32768 14.4 -> 14.0 (12.8); block 128 bf16 1000 x 5003 11.3 -> 9.8 (15.3), fp32 12.7 -> 10.7 (16.5)
// at 4097 x 1023.
// ALONE: there are no full tiles; the loads are non-temporal like theirs (see quantize_dual_ends).
// The workgroup's tiles: first_tile, first_tile + tile_step, ...
template <int DT, int B, bool ALIGNED, bool SUM, int NH, bool FULL, bool ALONE = false>
__device__ __forceinline__ void dual_tiles(DualLds<DT, B, SUM, NH> &lds, const void *__restrict__ x, int8_t *__restrict__ q, float *__restrict__ scales,
                                           int8_t *__restrict__ qT, float *__restrict__ scalesT, float *__restrict__ colsum_part, int64_t R, int64_t C, int64_t ldx,
                                           int64_t ldq, int64_t ldqt, int64_t Rp, int64_t Cp, int first_tile, int tile_step) {
    using L = DualLds<DT, B, SUM, NH>;
    constexpr int VEC = Bi8Vec<DT>::kElems;
    constexpr int ES = L::kES, CPT = L::kCPT, G = L::kG;
    constexpr int LPR = kTC / VEC;                 // lanes per half row: 8 (16-bit) or 16 (fp32)
    constexpr int RPP = kThreads / LPR;            // rows per load pass
    constexpr int NP = kTR / RPP;                  // load passes per half
    constexpr int NCORR = (DT == BI8_F32) ? 2 : 1;
    constexpr int RPT = kTR / G;                   // rows per thread in the column walk: 32 (fp32) or 16
    constexpr int GPW = B / RPT;                   // row groups per column block
    constexpr int LB = (B < kTC ? B : kTC) / VEC;  // lanes of one half row that share a row block
    constexpr int TC = NH * kTC;                   // columns of a tile
    static_assert(B == 32 || B == 64 || B == 128, "tile = one or more whole blocks in both directions");
    static_assert(NH == 2 || (NH == 1 && B <= kTC), "a row block lies inside the tile");
    static_assert(GPW > 1 || B == RPT, "a thread's rows are inside one block");

    const int tid = threadIdx.x;
    const bool wide_q = (((uintptr_t)q | (uintptr_t)ldq) & 15) == 0;     // rows of q on 16-byte boundaries: 16-byte code stores
    const int lr = tid / LPR;                      // row inside a pass
    const int cc = (tid % LPR) * VEC;              // first column of this lane inside a half

    const int full_r = (int)(R / kTR), full_c = (int)(C / TC);
    const int all_r = (int)((Rp + kTR - 1) / kTR), all_c = (int)((Cp + TC - 1) / TC);
    const int right = all_r * (all_c - full_c);    // tiles in the columns behind the full ones; then those below them
    const int ntiles = FULL ? full_r * full_c : right + (all_r - full_r) * full_c;
    auto coords = [&](int t, int &tr, int &tc) {
        if constexpr (FULL) {
            tile_coords<!ALIGNED>(t, full_r, full_c, tr, tc);
        } else if (t < right) {
            tr = t / (all_c - full_c);
            tc = full_c + t % (all_c - full_c);
        } else {
            tr = full_r + (t - right) / full_c;
            tc = (t - right) % full_c;
        }
    };
    constexpr bool kShift = !FULL && !ALIGNED;
    const char *x_lane = (const char *)x + ((int64_t)lr * ldx + cc) * ES;
    auto load_half = [&](int tr, int tc, int h, bi8_v4u *raw) {
        const int64_t r0 = (int64_t)tr * kTR, c0 = (int64_t)tc * TC + h * kTC;
        // a chunk that ends past a row's end is the row's last 16 bytes (see settle)
        const int64_t ahead = kShift && C >= VEC && c0 + cc > C - VEC ? c0 + cc - (C - VEC) : 0;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const char *src = x_lane + ((r0 + p * RPP) * ldx + c0 - ahead) * ES;
            if constexpr (FULL) {
                if constexpr (ALIGNED) raw[p] = __builtin_nontemporal_load((const bi8_v4u *)src);
                else raw[p] = *(const bi8_v4u_unaligned *)src;
            } else {
                raw[p] = bi8_v4u{0u, 0u, 0u, 0u};
                if (r0 + p * RPP + lr >= R || c0 + cc >= C) continue;
                if constexpr (ALIGNED) {
                    if constexpr (ALONE) raw[p] = __builtin_nontemporal_load((const bi8_v4u *)src);
                    else raw[p] = *(const bi8_v4u *)src;
                } else if (C >= VEC) {
                    raw[p] = *(const bi8_v4u_unaligned *)src;
                } else {                           // a row shorter than a chunk
#pragma unroll
                    for (int e = 0; e < VEC - 1; ++e) {
                        if (e < C) {
                            if constexpr (DT == BI8_F32) raw[p][e] = ((const uint32_t *)src)[e];
                            else raw[p][e >> 1] |= (uint32_t)((const uint16_t *)src)[e] << (16 * (e & 1));
                        }
                    }
                }
            }
        }
    };
    // ... of which the last `pieces` times 16 bits come to the front
    auto settle = [&](bi8_v4u v, int pieces) {
        if (pieces & 4) v = bi8_v4u{v[2], v[3], 0u, 0u};
        if (pieces & 2) v = bi8_v4u{v[1], v[2], v[3], 0u};
        if constexpr (ES == 2)
            if (pieces & 1) v = bi8_v4u{v[0] >> 16 | v[1] << 16, v[1] >> 16 | v[2] << 16, v[2] >> 16 | v[3] << 16, v[3] >> 16};
        return v;
    };

    if (first_tile >= ntiles) return;
    int tr, tc;
    coords(first_tile, tr, tc);
    bi8_v4u raw[NH][NP];
#pragma unroll
    for (int h = 0; h < NH; ++h) load_half(tr, tc, h, raw[h]);
    for (int tile = first_tile;;) {
        const int64_t r0 = (int64_t)tr * kTR, cbase = (int64_t)tc * TC;
        const int next = tile + tile_step;
        int tr_n = 0, tc_n = 0;
        if (next < ntiles) coords(next, tr_n, tc_n);
        const bool all_columns = FULL || cbase + TC <= Cp, all_rows = FULL || r0 + kTR <= Rp;      // ... of the tile are written
        int ahead[NH];                             // how far behind its chunk's first element a lane's load begins, in 16-bit pieces
        if constexpr (kShift) {
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                const int64_t n = cbase + h * kTC + cc - (C - VEC);
                ahead[h] = n > 0 && n < VEC && C >= VEC ? (int)n * (ES / 2) : 0;
            }
        }

        // ---- along the rows, from the registers ----------------------------------------------------------------
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const int64_t row = r0 + p * RPP + lr;
            if (!FULL && r0 + p * RPP >= R) break; // (nothing of these rows is stored)
            if constexpr (kShift) {
#pragma unroll
                for (int h = 0; h < NH; ++h)
                    if (__any(ahead[h] != 0)) raw[h][p] = settle(raw[h][p], ahead[h]);
            }
            uint32_t bits[NH];
            float m[NH];
            bi8_v2u wq[NH];                        // (fp32: four codes, the first word)
            bool slow = false;
#pragma unroll
            for (int h = 0; h < NH; ++h) bits[h] = bi8_magnitude_bits<DT>(raw[h][p]);
            if constexpr (B == 2 * kTC) {
                m[0] = m[NH - 1] = bi8_magnitude_of<DT>(bi8_group_bits<DT, LPR>(bi8_larger_bits<DT>(bits[0], bits[NH - 1])));
            } else {
#pragma unroll
                for (int h = 0; h < NH; ++h) m[h] = bi8_magnitude_of<DT>(bi8_group_bits<DT, LB>(bits[h]));
            }
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                float f[VEC];
                bi8_unpack<DT>(raw[h][p], f);
                slow |= !bi8_scale_is_fast(m[h]);
                const float y = bi8_recip_of_scale(m[h]);
                uint32_t code[VEC];
#pragma unroll
                for (int e = 0; e < VEC; ++e) code[e] = bi8_code_fast<NCORR>(f[e], m[h], y);
                wq[h][0] = bi8_pack4(code[0], code[1], code[2], code[3]);
                if constexpr (VEC == 8) wq[h][1] = bi8_pack4(code[4], code[5], code[6], code[7]);
            }
            if (__builtin_expect(__any(slow), 0)) {          // (the lanes of a block agree on it)
                float s[NH];
#pragma unroll
                for (int h = 0; h < NH; ++h) {
                    float f[VEC];
                    bi8_unpack<DT>(raw[h][p], f);
                    s[h] = 0.0f;
#pragma unroll
                    for (int e = 0; e < VEC; ++e) s[h] = __builtin_fmaxf(s[h], __builtin_fabsf(f[e]));     // ignores NaN
                }
                if constexpr (B == 2 * kTC) {
                    s[0] = s[NH - 1] = bi8_group_max<LPR>(__builtin_fmaxf(s[0], s[NH - 1]));
                } else {
#pragma unroll
                    for (int h = 0; h < NH; ++h) s[h] = bi8_group_max<LB>(s[h]);
                }
#pragma unroll
                for (int h = 0; h < NH; ++h) {
                    if (bi8_scale_is_fast(m[h])) continue;
                    float f[VEC];
                    bi8_unpack<DT>(raw[h][p], f);
                    m[h] = s[h];
                    uint32_t code[VEC];
#pragma unroll
                    for (int e = 0; e < VEC; ++e) code[e] = bi8_code_slow(f[e], s[h]);
                    wq[h][0] = bi8_pack4(code[0], code[1], code[2], code[3]);
                    if constexpr (VEC == 8) wq[h][1] = bi8_pack4(code[4], code[5], code[6], code[7]);
                }
            }
#pragma unroll
            for (int h = 0; h < NH; ++h)
                if ((tid % LB) == 0 && (B != 2 * kTC || h == 0)) lds.rs[(h * kTC + cc) / B][p * RPP + lr] = m[h];
            if (all_columns) {
                // (16-bit inputs, two halves: a lane's 8 codes of each half are exchanged with its neighbour's so that the
                // even lane stores 16 consecutive codes of the left half and the odd lane 16 of the right half -- the eight lanes of
                // a row then write the row's whole 128-byte line in one instruction instead of two halves in two; not in the tiles at
                // the matrix' ends, where it is the registers that spill)
                constexpr bool kPairs = VEC == 8 && NH == 2;
                if (wide_q && (FULL || !kPairs)) {
                    if constexpr (kPairs) {
                        const bool odd = (tid & 1) != 0;
                        const bi8_v2u send = odd ? wq[0] : wq[NH - 1];        // what the neighbour stores of this lane's codes
                        const bi8_v2u recv = {bi8_dpp_bits<0xB1>(send[0]), bi8_dpp_bits<0xB1>(send[1])};     // quad_perm [1,0,3,2]
                        const bi8_v4u w = odd ? bi8_v4u{recv[0], recv[1], wq[NH - 1][0], wq[NH - 1][1]} : bi8_v4u{wq[0][0], wq[0][1], recv[0], recv[1]};
                        __builtin_nontemporal_store(w, (bi8_v4u *)(q + row * ldq + cbase + (odd ? kTC + cc - VEC : cc)));
                    } else if (FULL || row < R) {
#pragma unroll
                        for (int h = 0; h < NH; ++h) {
                            int8_t *dst = q + row * ldq + cbase + h * kTC + cc;
                            if constexpr (VEC == 8) __builtin_nontemporal_store(wq[h], (bi8_v2u *)dst);
                            else __builtin_nontemporal_store(wq[h][0], (uint32_t *)dst);
                        }
                    }
                } else if (FULL || row < R) {
#pragma unroll
                    for (int h = 0; h < NH; ++h) {
                        int8_t *dst = q + row * ldq + cbase + h * kTC + cc;
                        if constexpr (VEC == 8) *(bi8_v2u_unaligned *)dst = wq[h];
                        else *(bi8_u32_unaligned *)dst = wq[h][0];
                    }
                }
            } else if (row < R) {
#pragma unroll
                for (int h = 0; h < NH; ++h) {
                    const int64_t col = cbase + h * kTC + cc;
                    int8_t *dst = q + row * ldq + col;
                    if (col + VEC <= Cp) {
                        if constexpr (VEC == 8) *(bi8_v2u_unaligned *)dst = wq[h];
                        else *(bi8_u32_unaligned *)dst = wq[h][0];
                    } else {
#pragma nounroll
                        for (int e = 0; e < (int)(Cp - col); ++e) dst[e] = (int8_t)((wq[h][VEC == 8 && e >= 4 ? 1 : 0] >> (8 * (e & 3))) & 0xffu);
                    }
                }
            }
        }

        // ---- down the columns, one half at a time through LDS --------------------------------------------------
#pragma unroll
        for (int h = 0; h < NH; ++h) {
            const int64_t c0 = cbase + h * kTC;
            // phase 1: this half -> LDS as it is (the previous half's column reads ended before the barrier that
            // precedes its phase 4); then start the next tile's loads of this half
#pragma unroll
            for (int p = 0; p < NP; ++p) *(bi8_v4u *)&lds.x[(p * RPP + lr) * L::kXPitch + (tid % LPR) * 16] = raw[h][p];
            if (FULL && next < ntiles) load_half(tr_n, tc_n, h, raw[h]);
            __syncthreads();
            if (h == 0) {
#pragma unroll
                for (int i = tid; i < L::kNRB * kTR; i += kThreads) {
                    const int b = i / kTR, r = i % kTR;
                    if (FULL || (r0 + r < R && cbase + b * B < Cp)) scales[(cbase / B + b) * R + r0 + r] = lds.rs[b][r];
                }
            }

            // phase 2: column maxima over this thread's rows (one 32-bit word column: one fp32 column or two 16-bit
            // columns), then over the block's row groups
            const int cw = tid % (kTC / CPT);
            const int g = tid / (kTC / CPT);
            uint32_t d[RPT];
#pragma unroll
            for (int i = 0; i < RPT; ++i) d[i] = *(const uint32_t *)&lds.x[(g * RPT + i) * L::kXPitch + cw * 4];
            uint32_t bits = bi8_abs_bits<DT>(d[0]);
#pragma unroll
            for (int i = 1; i < RPT; ++i) bits = bi8_larger_bits<DT>(bits, bi8_abs_bits<DT>(d[i]));
            if constexpr (SUM) {
                // this thread's rows of its columns, top to bottom (rows past R were loaded as zeros)
#pragma unroll
                for (int k = 0; k < CPT; ++k) {
                    float t = word_elem<DT>(d[0], k);
#pragma unroll
                    for (int i = 1; i < RPT; ++i) t += word_elem<DT>(d[i], k);
                    lds.sum[g][cw * CPT + k] = t;
                }
                // (the codes unpack the words again: kept from here they would be twice the registers)
#pragma unroll
                for (int i = 0; i < RPT; ++i) asm volatile("" : "+v"(d[i]));
            }
            if constexpr (GPW > 1 || SUM) {
                if constexpr (GPW > 1) lds.max[g][cw] = bits;
                __syncthreads();
                if constexpr (SUM) {
                    // the tile's row groups in ascending order; read before the barrier that follows phase 3, written
                    // again after the one that follows the next phase 1
                    if (g == 0) {
#pragma unroll
                        for (int k = 0; k < CPT; ++k) {
                            float t = lds.sum[0][cw * CPT + k];
#pragma unroll
                            for (int qg = 1; qg < G; ++qg) t += lds.sum[qg][cw * CPT + k];
                            if (FULL || c0 + cw * CPT + k < C) colsum_part[tr * C + c0 + cw * CPT + k] = t;
                        }
                    }
                }
                if constexpr (GPW > 1) {
                    const int gb = g & ~(GPW - 1);
                    bits = lds.max[gb][cw];
#pragma unroll
                    for (int qg = 1; qg < GPW; ++qg) bits = bi8_larger_bits<DT>(bits, lds.max[gb + qg][cw]);
                }
            }
            float mc[CPT];
            bool slow_c = false;
#pragma unroll
            for (int k = 0; k < CPT; ++k) mc[k] = word_elem<DT>(bits, k);

            // phase 3: codes of this thread's rows -> byte tile [column][row], 16 bytes per store
            bi8_v4u w[CPT][RPT / 16];
#pragma unroll
            for (int k = 0; k < CPT; ++k) {
                slow_c |= !bi8_scale_is_fast(mc[k]);
                const float y = bi8_recip_of_scale(mc[k]);
#pragma unroll
                for (int i = 0; i < RPT; i += 4) {
                    uint32_t code[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) code[e] = bi8_code_fast<NCORR>(word_elem<DT>(d[i + e], k), mc[k], y);
                    w[k][i / 16][(i % 16) / 4] = bi8_pack4(code[0], code[1], code[2], code[3]);
                }
            }
            if (__builtin_expect(__any(slow_c), 0)) {
#pragma unroll
                for (int k = 0; k < CPT; ++k) {
                    if (bi8_scale_is_fast(mc[k])) continue;
                    float s = 0.0f;                // of the block's rows, from the tile (the other groups' maxima hold its NaNs)
#pragma nounroll
                    for (int r = g * RPT / B * B; r < g * RPT / B * B + B; ++r)
                        s = __builtin_fmaxf(s, __builtin_fabsf(word_elem<DT>(*(const uint32_t *)&lds.x[r * L::kXPitch + cw * 4], k)));
                    mc[k] = s;
#pragma unroll
                    for (int i = 0; i < RPT; i += 4) {
                        uint32_t code[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) code[e] = bi8_code_slow(word_elem<DT>(d[i + e], k), s);
                        w[k][i / 16][(i % 16) / 4] = bi8_pack4(code[0], code[1], code[2], code[3]);
                    }
                }
            }
            if ((g & (GPW - 1)) == 0) {
                const int64_t jb = (r0 + g * RPT) / B;
#pragma unroll
                for (int k = 0; k < CPT; ++k)
                    if (FULL || (r0 + g * RPT < Rp && c0 + cw * CPT + k < C)) scalesT[jb * C + c0 + cw * CPT + k] = mc[k];
            }
#pragma unroll
            for (int k = 0; k < CPT; ++k)
#pragma unroll
                for (int i = 0; i < RPT / 16; ++i) *(bi8_v4u *)&lds.q[(cw * CPT + k) * kQPitch + g * RPT + 16 * i] = w[k][i];
            __syncthreads();

            // phase 4: 16 codes per lane, 8 lanes per output row.  The next writes to the tile come after this barrier, the
            // next writes to the code tile after the next phase-1 barrier.
#pragma unroll
            for (int p = 0; p < (kTC * kTR / 16) / kThreads; ++p) {
                const int idx = p * kThreads + tid;
                const int oc = idx / (kTR / 16);       // output row inside the half = source column
                const int seg = idx % (kTR / 16);
                const int64_t orow = c0 + oc;
                const int64_t ocol = r0 + seg * 16;
                const bi8_v4u v = *(const bi8_v4u *)&lds.q[oc * kQPitch + seg * 16];
                int8_t *dst = qT + orow * ldqt + ocol;
                if (all_rows) {
                    if (FULL || orow < C) __builtin_nontemporal_store(v, (bi8_v4u *)dst);
                } else if (orow < C && ocol + 16 <= Rp) {
                    *(bi8_v4u *)dst = v;
                } else if (orow < C) {
#pragma nounroll
                    for (int e = 0; e < (int)(Rp - ocol); ++e) dst[e] = (int8_t)((v[e >> 2] >> (8 * (e & 3))) & 0xffu);
                }
            }
        }
        if (next >= ntiles) break;
        tile = next;
        tr = tr_n;
        tc = tc_n;
        if constexpr (!FULL) {                     // (a workgroup rarely has two of these: not under the tile before, which would spill)
#pragma unroll
            for (int h = 0; h < NH; ++h) load_half(tr, tc, h, raw[h]);
        }
    }
}

// All of a matrix' tiles: workgroup `first` of `step` takes every step-th of the full ones, then of the others, counted on from there.
template <int DT, int B, bool ALIGNED, bool SUM, int NH>
__device__ __forceinline__ void dual_matrix(const Bi8DualTask &t, float *colsum_part, int first, int step) {
    __shared__ DualLds<DT, B, SUM, NH> lds;
    dual_tiles<DT, B, ALIGNED, SUM, NH, true>(lds, t.x, t.q, t.scales, t.qT, t.scalesT, colsum_part, t.R, t.C, t.ldx, t.ldq, t.ldqt, t.Rp, t.Cp, first, step);
    if (t.Rp % kTR == 0 && t.Cp % (NH * kTC) == 0 && t.Rp == t.R && t.Cp == t.C) return;
    const int full = (int)(t.R / kTR) * (int)(t.C / (NH * kTC));
    const int offset = (first - full % step + step) % step;
    __syncthreads();                               // the last full tile has been read
    dual_tiles<DT, B, ALIGNED, SUM, NH, false>(lds, t.x, t.q, t.scales, t.qT, t.scalesT, colsum_part, t.R, t.C, t.ldx, t.ldq, t.ldqt, t.Rp, t.Cp, offset, step);
}

#define BI8_DUAL_KERNEL __global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(DT == BI8_F32 ? 3 : 4)))
template <int DT, int B, bool ALIGNED, bool SUM, int NH>
BI8_DUAL_KERNEL void quantize_dual_tile(const Bi8DualTask task, float *__restrict__ colsum_part) {
    dual_matrix<DT, B, ALIGNED, SUM, NH>(task, colsum_part, blockIdx.x, gridDim.x);
}

// A matrix without a full tile (fewer than 128 rows, say), its rows on 16-byte boundaries.  us, by the kernel above with plain loads -> this: block 64 fp32
// 16 x 4096 4.2 -> 4.0, 100 x 32768 9.2 -> 8.2, 120 x 8192 6.8 -> 6.3, bf16 100 x 32768 7.2 -> 6.6, 100 x 11008 5.3 -> 5.0; block 128 fp32 100 x 11008
// 8.9 -> 8.2, bf16 100 x 32768 9.0 -> 8.2.
// Not under full tiles' kernels: there it costs fp32 with column sums up to six more spilled registers (4096 x 4096, block 64 25.3 -> 27.0), and
// behind full tiles non-temporal loads lose (fp32 500 x 16384 14.7 -> 15.1).  No such kernel with column sums.
template <int DT, int B, int NH> BI8_DUAL_KERNEL void quantize_dual_ends(const Bi8DualTask t) {
    __shared__ DualLds<DT, B, false, NH> lds;
    dual_tiles<DT, B, true, false, NH, false, true>(lds, t.x, t.q, t.scales, t.qT, t.scalesT, nullptr, t.R, t.C, t.ldx, t.ldq, t.ldqt, t.Rp, t.Cp, blockIdx.x, gridDim.x);
}

// Two matrices: the grid's first blocks0 workgroups work on the first, the others on the second (a layer's X and W: one launch, and
// the smaller of the two does not have the chip to itself half empty).
struct DualPair {
    Bi8DualTask task[2];
    unsigned blocks0;
};
template <int DT, int B, bool ALIGNED, int NH> BI8_DUAL_KERNEL void quantize_dual_pair(const DualPair pair) {
    const bool second = blockIdx.x >= pair.blocks0;
    const Bi8DualTask &t0 = pair.task[0], &t1 = pair.task[1];
#define BI8_OF_TASK(f) (second ? t1.f : t0.f)
    const Bi8DualTask task{BI8_OF_TASK(x), BI8_OF_TASK(q), BI8_OF_TASK(qT), BI8_OF_TASK(scales), BI8_OF_TASK(scalesT), BI8_OF_TASK(R), BI8_OF_TASK(C),
                           BI8_OF_TASK(ldx), BI8_OF_TASK(ldq), BI8_OF_TASK(ldqt), BI8_OF_TASK(Rp), BI8_OF_TASK(Cp)};
#undef BI8_OF_TASK
    dual_matrix<DT, B, ALIGNED, false, NH>(task, nullptr, (int)(second ? blockIdx.x - pair.blocks0 : blockIdx.x), (int)(second ? gridDim.x - pair.blocks0 : pair.blocks0));
}

template <int DT, int B, bool ALIGNED, int NH> int launch_one(const Bi8DualTask &t, float *colsum_part, int64_t resident, hipStream_t st) {
    const int64_t ntiles = ((t.Cp + NH * kTC - 1) / (NH * kTC)) * ((t.Rp + kTR - 1) / kTR);
    if (ntiles + resident > 0x7fffffffLL) return BI8_ERR_TOO_LARGE;
    const dim3 grid((unsigned)(ntiles < resident ? ntiles : resident));
    if constexpr (ALIGNED) {
        if (!colsum_part && (t.R < kTR || t.C < NH * kTC)) {
            hipLaunchKernelGGL((quantize_dual_ends<DT, B, NH>), grid, dim3(kThreads), 0, st, t);
            return bi8_launch_rc();
        }
    }
    if (colsum_part) hipLaunchKernelGGL((quantize_dual_tile<DT, B, ALIGNED, true, NH>), grid, dim3(kThreads), 0, st, t, colsum_part);
    else hipLaunchKernelGGL((quantize_dual_tile<DT, B, ALIGNED, false, NH>), grid, dim3(kThreads), 0, st, t, colsum_part);
    return bi8_launch_rc();
}

// Both matrices in one launch, the resident workgroups in proportion to the tiles; BI8_ERR_UNSUPPORTED where that is not taken: from kPairRounds
// rounds of workgroups on it has to save one.  The mixed traffic of two matrices costs about 1 % (bf16, block 128, X 4096 x 4096 and W
// 11008 x 4096, 1024 and 2752 tiles, four rounds either way: 55.6 us in two launches, 56.6 in one; in a training pass 668 against 672), the
// second launch about 1.5 us.  us, two launches -> one, tiles of X + W and rounds: 48 + 108 (2 -> 1) 12.2 -> 7.0; 1024 + 1024 (2 -> 2) 31.8 ->
// 30.3; at fp32 (768 workgroups) 1710 + 665 (4 -> 4) 67.7 -> 67.7, 672 + 1120 (3 -> 3) 50.1 -> 49.6; 1836 + 4104 (7 -> 6) 92.1 -> 84.4.
constexpr int64_t kPairRounds = 4;
template <int DT, int B, bool ALIGNED, int NH> int launch_pair(const Bi8DualTask *task, int64_t resident, hipStream_t st) {
    DualPair pair{{task[0], task[1]}, 0};
    int64_t tiles[2];
    for (int i = 0; i < 2; ++i) tiles[i] = ((task[i].Cp + NH * kTC - 1) / (NH * kTC)) * ((task[i].Rp + kTR - 1) / kTR);
    const int64_t all = tiles[0] + tiles[1], grid = all < resident ? all : resident;
    if (all + resident > 0x7fffffffLL) return BI8_ERR_TOO_LARGE;
    int64_t first = all <= resident ? tiles[0] : (grid * tiles[0] + all / 2) / all;
    first = first < 1 ? 1 : first > grid - 1 ? grid - 1 : first;
    const int64_t apart = (tiles[0] + resident - 1) / resident + (tiles[1] + resident - 1) / resident;
    const int64_t r0 = (tiles[0] + first - 1) / first, r1 = (tiles[1] + grid - first - 1) / (grid - first);
    if (apart >= kPairRounds && (r0 > r1 ? r0 : r1) >= apart) return BI8_ERR_UNSUPPORTED;
    pair.blocks0 = (unsigned)first;
    hipLaunchKernelGGL((quantize_dual_pair<DT, B, ALIGNED, NH>), dim3((unsigned)grid), dim3(kThreads), 0, st, pair);
    return bi8_launch_rc();
}

// Whole tiles also where that is two for each CU and not a third but at the matrix' ends: as half tiles those at the ends are a workgroup's
// second ones, which are not loaded under the first.  us, half / whole (before the two kinds of tiles; half ones), block 64: bf16 300 x 32768
// 13.7 / 12.2 (12.8), 1000 x 8192 11.3 / 10.5 (11.5), 8192 x 1000 13.4 / 12.2 (13.6), 2048 x 4096 10.9 / 10.3 (11.0), 700 x 12288 12.4 / 11.7 (12.8), two of 1000 x
// 4096 11.6 / 10.3 (10.8); fp32 8192 x 1000 16.7 / 16.0 (15.8), 500 x 16384 14.5 / 14.3 (14.5), 700 x 12288 16.0 / 15.6 (16.2).  With fewer elements (300 x 24576
// bf16 11.2 / 11.6, fp32 13.9 / 15.0), a third tile (11008 x 768 bf16 11.2 / 12.1, fp32 15.1 / 17.1; 1000 x 11008 bf16 14.2 / 14.4), rows off 16-byte boundaries
// (2000 x 5003 14.8 / 15.2, fp32 18.7 / 20.6), fp32 without ends (4096 x 2048 13.8 / 14.0) or with column sums (8192 x 1024 13.7 / 14.4): half ones.
constexpr int64_t kTwoEachElems = 8000000;
template <int DT, int B, bool ALIGNED> int launch_dual(const Bi8DualTask *task, int count, float *colsum_part, hipStream_t st) {
    // workgroups per CU: four with 16-bit inputs (30 KiB of LDS, at most 128 registers), three with fp32 (43 KiB, 168).  us with three
    // / four: bf16 [8192,4096] 29.5 / 28.6, [8192,3072] 22.7 / 22.7, fp32 [4096,4096] 23.5 / 27.9
    const int64_t resident = (DT == BI8_F32 ? 3 : 4) * 256;
    // inputs of fewer full tiles than the chip holds workgroups: half tiles, twice as many workgroups
    int64_t full = 0, inside = 0, elems = 0;
    for (int i = 0; i < count; ++i) {
        full += ((task[i].Cp + 2 * kTC - 1) / (2 * kTC)) * ((task[i].Rp + kTR - 1) / kTR);
        inside += (task[i].C / (2 * kTC)) * (task[i].R / kTR);
        elems += task[i].R * task[i].C;
    }
    constexpr int kHalf = B <= kTC ? 1 : 2;
    const bool two_each = ALIGNED && elems >= kTwoEachElems && inside <= 2 * 256 && (DT != BI8_F32 || (!colsum_part && inside < full));
    const bool half = full < resident && !two_each;
    if (count == 1)
        return half ? launch_one<DT, B, ALIGNED, kHalf>(task[0], colsum_part, resident, st) : launch_one<DT, B, ALIGNED, 2>(task[0], colsum_part, resident, st);
    const int rc = half ? launch_pair<DT, B, ALIGNED, kHalf>(task, resident, st) : launch_pair<DT, B, ALIGNED, 2>(task, resident, st);
    if (rc != BI8_ERR_UNSUPPORTED) return rc;
    const int rc0 = launch_dual<DT, B, ALIGNED>(task, 1, nullptr, st);
    return rc0 != BI8_OK ? rc0 : launch_dual<DT, B, ALIGNED>(task + 1, 1, nullptr, st);
}

template <int DT, bool ALIGNED> int dispatch(const Bi8DualTask *task, int count, float *colsum_part, int block, hipStream_t st) {
    switch (block) {
    case 32: return launch_dual<DT, 32, ALIGNED>(task, count, colsum_part, st);
    case 64: return launch_dual<DT, 64, ALIGNED>(task, count, colsum_part, st);
    default: return launch_dual<DT, 128, ALIGNED>(task, count, colsum_part, st);
    }
}

}  // namespace

// This file is compiled once per input type with -DBI8_DUAL_DT=d, which gives the one function below with that type's kernels, and once
// without for everything else: one translation unit with all of them takes two minutes.
#define BI8_DUAL_RUN_PASTE(d) bi8_dual_run_##d
#define BI8_DUAL_RUN_NAME(d) BI8_DUAL_RUN_PASTE(d)
#define BI8_DUAL_RUN(d) int BI8_DUAL_RUN_NAME(d)(const Bi8DualTask *task, int count, bool aligned, float *colsum_part, int block, hipStream_t st)
#ifdef BI8_DUAL_DT
__attribute__((visibility("hidden"))) BI8_DUAL_RUN(BI8_DUAL_DT) {
    return aligned ? dispatch<BI8_DUAL_DT, true>(task, count, colsum_part, block, st) : dispatch<BI8_DUAL_DT, false>(task, count, colsum_part, block, st);
}
#else
BI8_DUAL_RUN(0);
BI8_DUAL_RUN(1);
BI8_DUAL_RUN(2);
static_assert(BI8_F32 == 0 && BI8_BF16 == 1 && BI8_F16 == 2, "the names of the functions");

namespace {

// Column sums without the quantizer (the shapes that the one-pass kernel does not take): the same grouping of the
// rows -- groups of kTR / G rows top to bottom, the groups of a 128-row tile in ascending order -- so that the sums
// do not depend on which kernel made them.  One thread per column.
template <int DT>
__global__ __launch_bounds__(256) void colsum_tiles(const void *__restrict__ x, float *__restrict__ part, int64_t R, int64_t C, int64_t ldx) {
    constexpr int RPT = (DT == BI8_F32) ? 32 : 16;
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t tr = blockIdx.y;
    if (c >= C) return;
    float total = 0.0f;
    for (int g = 0; g < kTR / RPT; ++g) {
        float t = 0.0f;
        for (int i = 0; i < RPT; ++i) {
            const int64_t r = tr * kTR + g * RPT + i;
            const float v = r < R ? bi8_load_elem<DT>(x, r * ldx + c) : 0.0f;
            t = i == 0 ? v : t + v;
        }
        total = g == 0 ? t : total + t;
    }
    part[tr * C + c] = total;
}

// out[c] = cast(sum over the row tiles, ascending)
template <int DT>
__global__ __launch_bounds__(256) void colsum_finish(const float *__restrict__ part, void *__restrict__ out, int64_t tiles_r, int64_t C) {
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
    bi8_store_elem<DT>(out, c, bi8_sum_of_tiles(part, tiles_r, C, c));
}

template <int DT> int launch_colsum_finish(const float *part, void *out, int64_t tiles_r, int64_t C, hipStream_t st) {
    hipLaunchKernelGGL((colsum_finish<DT>), dim3((unsigned)((C + 255) / 256)), dim3(256), 0, st, part, out, tiles_r, C);
    return bi8_launch_rc();
}
template <int DT> int launch_colsum_tiles(const void *x, float *part, int64_t R, int64_t C, int64_t ldx, hipStream_t st) {
    const int64_t tiles_r = (R + kTR - 1) / kTR;
    if (tiles_r > 65535) return BI8_ERR_TOO_LARGE;
    hipLaunchKernelGGL((colsum_tiles<DT>), dim3((unsigned)((C + 255) / 256), (unsigned)tiles_r), dim3(256), 0, st, x, part, R, C, ldx);
    return bi8_launch_rc();
}

}  // namespace

// One kernel: block 32 / 64 / 128, x aligned to its element type, the transposed codes in 16-byte aligned rows.
static bool one_pass(const Bi8DualTask &t, int x_dtype, int block) {
    return (block == 32 || block == 64 || block == 128) && bi8_aligned(t.x, x_dtype == BI8_F32 ? 4 : 2) && t.ldqt % 16 == 0 && bi8_aligned(t.qT, 16);
}

extern "C" int bi8x_quantize_dual(const Bi8DualTask *task, int count, int x_dtype, int block, float *colsum_part, void *stream) {
    if (count < 1 || count > 2 || (count == 2 && colsum_part)) return BI8_ERR_BAD_SHAPE;
    const int64_t vec = x_dtype == BI8_F32 ? 4 : 8;
    bool aligned = true;
    for (int i = 0; i < count; ++i) {
        const Bi8DualTask &t = task[i];
        if (!one_pass(t, x_dtype, block)) return BI8_ERR_UNSUPPORTED;
        if (t.R < 1 || t.C < 1 || t.ldx < t.C || t.Cp < t.C || t.Rp < t.R || t.ldq < t.Cp || t.ldqt < t.Rp) return BI8_ERR_BAD_SHAPE;
        aligned = aligned && t.C % vec == 0 && t.ldx % vec == 0 && bi8_aligned(t.x, 16);
    }
    hipStream_t st = (hipStream_t)stream;
    switch (x_dtype) {
    case BI8_F32: return BI8_DUAL_RUN_NAME(0)(task, count, aligned, colsum_part, block, st);
    case BI8_BF16: return BI8_DUAL_RUN_NAME(1)(task, count, aligned, colsum_part, block, st);
    default: return BI8_DUAL_RUN_NAME(2)(task, count, aligned, colsum_part, block, st);
    }
}

static int quantize_dual(const void *x, int x_dtype, int8_t *q, float *scales, int8_t *qT, float *scalesT, float *colsum_part, int64_t R,
                         int64_t C, int64_t ldx, int64_t ldq, int64_t ldqt, int block, void *stream) {
    if (x_dtype < 0 || x_dtype > 2) return BI8_ERR_BAD_DTYPE;
    if (block < 1 || block > (1 << 20)) return BI8_ERR_BAD_BLOCK;
    if (R < 0 || C < 0 || ldx < C || ldq < C || ldqt < R) return BI8_ERR_BAD_SHAPE;
    if (R == 0 || C == 0) return BI8_OK;
    if (!x || !q || !scales || !qT || !scalesT) return BI8_ERR_NULL_POINTER;
    const Bi8DualTask task{x, q, qT, scales, scalesT, R, C, ldx, ldq, ldqt, R, C};
    if (!one_pass(task, x_dtype, block)) {
        // other block sizes, transposed rows of odd length: the two single-direction entry points, same results
        int rc = bi8_quantize_rowwise(x, x_dtype, q, scales, R, C, ldx, ldq, block, stream);
        if (rc != BI8_OK) return rc;
        rc = bi8_quantize_transposed(x, x_dtype, qT, scalesT, R, C, ldx, ldqt, block, stream);
        if (rc != BI8_OK || !colsum_part) return rc;
        switch (x_dtype) {
        case BI8_F32: return launch_colsum_tiles<BI8_F32>(x, colsum_part, R, C, ldx, (hipStream_t)stream);
        case BI8_BF16: return launch_colsum_tiles<BI8_BF16>(x, colsum_part, R, C, ldx, (hipStream_t)stream);
        default: return launch_colsum_tiles<BI8_F16>(x, colsum_part, R, C, ldx, (hipStream_t)stream);
        }
    }
    return bi8x_quantize_dual(&task, 1, x_dtype, block, colsum_part, stream);
}

extern "C" int bi8x_colsum_finish(const float *part, void *out, int dtype, int64_t R, int64_t C, void *stream) {
    const int64_t tiles_r = (R + kTR - 1) / kTR;
    switch (dtype) {
    case BI8_F32: return launch_colsum_finish<BI8_F32>(part, out, tiles_r, C, (hipStream_t)stream);
    case BI8_BF16: return launch_colsum_finish<BI8_BF16>(part, out, tiles_r, C, (hipStream_t)stream);
    default: return launch_colsum_finish<BI8_F16>(part, out, tiles_r, C, (hipStream_t)stream);
    }
}

extern "C" int bi8_quantize_dual(const void *x, int x_dtype, int8_t *q, float *scales, int8_t *qT, float *scalesT, int64_t R, int64_t C,
                                 int64_t ldx, int64_t ldq, int64_t ldqt, int block, void *stream) {
    return quantize_dual(x, x_dtype, q, scales, qT, scalesT, nullptr, R, C, ldx, ldq, ldqt, block, stream);
}

extern "C" int64_t bi8_colsum_workspace_bytes(int64_t R, int64_t C) {
    if (R <= 0 || C <= 0) return 0;
    return ((R + kTR - 1) / kTR) * C * (int64_t)sizeof(float);
}

extern "C" int bi8_quantize_dual_colsum(const void *x, int x_dtype, int8_t *q, float *scales, int8_t *qT, float *scalesT, void *colsum,
                                        void *workspace, int64_t workspace_bytes, int64_t R, int64_t C, int64_t ldx, int64_t ldq,
                                        int64_t ldqt, int block, void *stream) {
    if (x_dtype < 0 || x_dtype > 2) return BI8_ERR_BAD_DTYPE;
    if (R < 0 || C < 0) return BI8_ERR_BAD_SHAPE;
    if (C == 0) return BI8_OK;
    if (!colsum) return BI8_ERR_NULL_POINTER;
    if (R == 0) return bi8x_colsum_finish(nullptr, colsum, x_dtype, 0, C, stream);     // an empty sum: zeros
    if (!workspace || !bi8_aligned(workspace, 4)) return BI8_ERR_NULL_POINTER;
    if (workspace_bytes < bi8_colsum_workspace_bytes(R, C)) return BI8_ERR_BAD_SHAPE;
    const int rc = quantize_dual(x, x_dtype, q, scales, qT, scalesT, (float *)workspace, R, C, ldx, ldq, ldqt, block, stream);
    return rc != BI8_OK ? rc : bi8x_colsum_finish((const float *)workspace, colsum, x_dtype, R, C, stream);
}
#endif  // BI8_DUAL_DT
