// The offset terms of weight types that are held in another type's planes.
//
// The m * s term of the Q4_1 / Q5_1 dot product with Q8_1 activations (k_quants.rs:267-294, :463-494):
//   y[r, c] += sum_b  h2f(m[c, b]) * h2f(s8[r, b]),   s8 = f16(h2f(f16(sum of the block's 32 quants)) * d8)
// (BlockQ8_1::from_float, k_quants.rs:665-691).  Those weights are held as Q8_0 planes (quants 0..15 / 0..31) plus the
// plane of minima; the Q8_0 kernels have already written sum_b sum_i * d * d8 into y, from activations quantized by the
// Q8_0 rule, which is the Q8_1 rule without the `s` field: the field is recomputed here from the workspace's block sums
// and scales.  The reference adds both terms block by block into one f32; here the two sums are formed separately and
// added, a difference of rounding only.
#include "qhip_internal.h"

namespace {

__device__ __forceinline__ float block_s(const cq_act_view &a, int64_t at) {
    const float hs = cq_h2f(cq_f2h((float)a.bsum32[at]));
    return cq_h2f(cq_f2h(hs * a.d[at]));
}

typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// ---- many rows: the sums over blocks as products on the matrix cores ----
// Both factors of the m * s term are f16 values and their product is exact in f32; so are Q2K's integer sums, at most 16 * 2048 * 15.
// MFMA 32x32x16 (f16): lane l holds row l % 32 of either operand, k = 8 * (l / 32) .. + 7, and of the result column l % 32, rows
// 8 * (i / 4) + 4 * (l / 32) + i % 4.  Activation rows are the rows, weight rows the columns, so that a wave's stores are runs of 128 bytes.
// No LDS and no barrier: the operands are a few hundred bytes a row, read straight into registers (cache hits after the first tile); what
// is left is the pass over y and, with few tiles, a chain of loads.  Against the sums on the vector units through LDS, us a whole call before
// and after: Q5_1 2225 x 3328 with 3343 rows 187 -> 127, Q4_1 14336 x 4096 with 512 rows 184 -> 134, 4096 x 4096 with 64 rows 36.0 -> 21.2,
// Q2K 4096 x 4096 with 1024 rows 147 -> 88, with 128 rows 59.9 -> 28.7 (few rows: the split-K kernels add the terms themselves, skinny.hip).  Error of the m * s term against 64 bits
// (4096 x 4096, 64 rows, relative rms): 8.9e-8 -> 6.0e-8.
//   SHARE = false: every wave a 64 x 64 tile of its own (workgroup: 64 rows x 256 weight rows)
//   SHARE = true:  up to 32 rows x 32 weight rows a workgroup, the steps dealt round-robin to its four waves: few rows leave too few tiles to
//                  fill the machine, and one wave would walk the whole row by itself
struct HalfRow { uint32_t w[4]; };   // eight 16-bit values; rows have an even number of blocks and so start on a word
__device__ __forceinline__ HalfRow load_eight(const void *plane, int64_t row, int64_t b, int64_t nb) {
    const uint32_t *p = (const uint32_t *)plane + ((row * nb + b) >> 1);
    HalfRow r;
    if (b + 8 <= nb) {
#pragma unroll
        for (int i = 0; i < 4; i++) r.w[i] = p[i];
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) r.w[i] = b + 2 * i < nb ? p[i] : 0u;
    }
    return r;
}

// Adds (or, SUB, subtracts) the tile to y; SHARE: the four waves' parts first, in order.
template <bool SHARE, bool SUB, int RT, int CT>
__device__ __forceinline__ void add_tiles(v16f (&acc)[RT][CT], int64_t r0, int64_t c0, int64_t m, int64_t n, float *__restrict__ y) {
    const int lane = threadIdx.x & 63, col = lane & 31, h = lane >> 5;
    if constexpr (SHARE) {
        __shared__ float part[4][16][64];
        const int wave = threadIdx.x >> 6;
#pragma unroll
        for (int i = 0; i < 16; i++) part[wave][i][lane] = acc[0][0][i];
        __syncthreads();
        if (c0 + col >= n) return;
#pragma unroll
        for (int j = 0; j < 4; j++) {   // wave w finishes result registers 4w .. 4w + 3
            const int i = 4 * wave + j;
            const int64_t r = r0 + 8 * wave + 4 * h + j;
            const float t = ((part[0][i][lane] + part[1][i][lane]) + part[2][i][lane]) + part[3][i][lane];
            if (r < m) y[r * n + c0 + col] += SUB ? -t : t;
        }
    } else {
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int ct = 0; ct < CT; ct++) {
                const int64_t c = c0 + 32 * ct + col;
                float old[16];
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int64_t r = r0 + 32 * rt + 8 * (i >> 2) + 4 * h + (i & 3);
                    if (r < m && c < n) old[i] = y[r * n + c];
                }
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int64_t r = r0 + 32 * rt + 8 * (i >> 2) + 4 * h + (i & 3);
                    if (r < m && c < n) y[r * n + c] = old[i] + (SUB ? -acc[rt][ct][i] : acc[rt][ct][i]);
                }
            }
    }
}

template <bool SHARE>
__global__ void __launch_bounds__(256) min32_mfma_kernel(const uint16_t *__restrict__ mins, cq_act_view a, int64_t n, int64_t nb, int64_t m,
                                                         float *__restrict__ y) {
    constexpr int RT = SHARE ? 1 : 2, CT = SHARE ? 1 : 2;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, h = lane >> 5;
    const int64_t r0 = (int64_t)blockIdx.y * 32 * RT, c0 = ((int64_t)blockIdx.x * (SHARE ? 1 : 4) + (SHARE ? 0 : wave)) * 32 * CT;
    v16f acc[RT][CT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int ct = 0; ct < CT; ct++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[rt][ct][i] = 0.0f;
    int64_t rows[RT], cols[CT];   // (rows and weight rows past the end repeat the last one; their results are not stored)
#pragma unroll
    for (int rt = 0; rt < RT; rt++) rows[rt] = r0 + 32 * rt + (lane & 31) < m ? r0 + 32 * rt + (lane & 31) : m - 1;
#pragma unroll
    for (int ct = 0; ct < CT; ct++) cols[ct] = c0 + 32 * ct + (lane & 31) < n ? c0 + 32 * ct + (lane & 31) : n - 1;
    if (SHARE || c0 < n) {
        for (int64_t b0 = SHARE ? 16 * wave : 0; b0 < nb; b0 += SHARE ? 64 : 16) {
            const int64_t b = b0 + 8 * h;
            v8h mv[CT], sv[RT];
#pragma unroll
            for (int ct = 0; ct < CT; ct++) mv[ct] = __builtin_bit_cast(v8h, load_eight(mins, cols[ct], b, nb));
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
                const HalfRow sums = load_eight(a.bsum32, rows[rt], b, nb);
                const float *d = a.d + rows[rt] * nb + b;
                float dv[8];
                if (b + 8 <= nb) {
#pragma unroll
                    for (int i = 0; i < 8; i++) dv[i] = d[i];
                } else {
#pragma unroll
                    for (int i = 0; i < 8; i++) dv[i] = b + i < nb ? d[i] : 0.0f;
                }
#pragma unroll
                for (int i = 0; i < 8; i++) {   // (blocks past the end: both factors zero)
                    const float hs = (float)(_Float16)(float)(int16_t)(sums.w[i >> 1] >> (16 * (i & 1)));
                    sv[rt][i] = (_Float16)(hs * dv[i]);
                }
            }
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
#pragma unroll
                for (int ct = 0; ct < CT; ct++) acc[rt][ct] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sv[rt], mv[ct], acc[rt][ct], 0, 0, 0);
        }
    }
    add_tiles<SHARE, false, RT, CT>(acc, r0, c0, m, n, y);
}

// Few rows (decode, small batches): sixteen lanes per weight row, each a chunk of eight blocks out of 128 at a time; lane
// 0 of the sixteen adds the chunk sums in order.  Sixteen weight rows and four activation rows per workgroup.
constexpr int kChunk = 8;
constexpr int kSmallRows = 4;
__global__ void __launch_bounds__(256) min32_small_kernel(const uint16_t *__restrict__ mins, cq_act_view a, int64_t n, int64_t nb,
                                                          int64_t m, float *__restrict__ y) {
    __shared__ float part[kSmallRows][16][17];
    const int j = threadIdx.x & 15, cl = threadIdx.x >> 4;
    const int64_t c = (int64_t)blockIdx.x * 16 + cl;
    const uint16_t *mrow = mins + (c < n ? c : n - 1) * nb;
    const int64_t r0 = (int64_t)blockIdx.y * kSmallRows;
    float acc[kSmallRows] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int64_t sb = 0; sb < nb; sb += 16 * kChunk) {
        const int64_t b = sb + j * kChunk;
        const int cnt = (int)(nb - b < kChunk ? (nb - b < 0 ? 0 : nb - b) : kChunk);
        float mv[kChunk];
#pragma unroll
        for (int i = 0; i < kChunk; i++) mv[i] = i < cnt ? cq_h2f(mrow[b + i]) : 0.0f;
#pragma unroll
        for (int r = 0; r < kSmallRows; r++) {
            float t = 0.0f;
            if (r0 + r < m) {
#pragma unroll
                for (int i = 0; i < kChunk; i++)
                    if (i < cnt) t += mv[i] * block_s(a, (r0 + r) * nb + b + i);
            }
            part[r][cl][j] = t;
        }
        __syncthreads();
        if (j == 0) {
            for (int jj = 0; jj < 16 && sb + jj * kChunk < nb; jj++)
#pragma unroll
                for (int r = 0; r < kSmallRows; r++) acc[r] += part[r][cl][jj];
        }
        __syncthreads();
    }
    if (j == 0 && c < n)
        for (int r = 0; r < kSmallRows && r0 + r < m; r++) y[(r0 + r) * n + c] += acc[r];
}

// ---- Q2K: the dmin term of its dot product with Q8K activations (k_quants.rs:727-733, :762) ----
//   y[r, c] -= sum_b (d8[r, b] * h2f(dmin[c, b])) * float(sum_j bsums[r, b, j] * m[c, b, j])
// Many rows: a block's sixteen products are one MFMA step, its result the exact integer; scaled and added block by block.
template <bool SHARE>
__global__ void __launch_bounds__(256) min16_mfma_kernel(const uint8_t *__restrict__ mins, const uint16_t *__restrict__ dmins, cq_act_view a,
                                                         int64_t n, int64_t kb, int64_t m, float *__restrict__ y) {
    constexpr int RT = SHARE ? 1 : 2, CT = SHARE ? 1 : 2;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, h = lane >> 5;
    const int64_t r0 = (int64_t)blockIdx.y * 32 * RT, c0 = ((int64_t)blockIdx.x * (SHARE ? 1 : 4) + (SHARE ? 0 : wave)) * 32 * CT;
    v16f acc[RT][CT];
    v16f zero;
#pragma unroll
    for (int i = 0; i < 16; i++) zero[i] = 0.0f;
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int ct = 0; ct < CT; ct++) acc[rt][ct] = zero;
    int64_t cols[CT];   // (weight rows past the end repeat the last one; rows past the end are the workspace's padding; neither is stored)
#pragma unroll
    for (int ct = 0; ct < CT; ct++) cols[ct] = c0 + 32 * ct + (lane & 31) < n ? c0 + 32 * ct + (lane & 31) : n - 1;
    if (SHARE || c0 < n) {
        for (int64_t b = SHARE ? wave : 0; b < kb; b += SHARE ? 4 : 1) {
            v8h mv[CT], sv[RT];
            float dm[CT];
            const _Float16 k1024 = (_Float16)1024.0f;
#pragma unroll
            for (int ct = 0; ct < CT; ct++) {
                const uint2 w = *(const uint2 *)(mins + (cols[ct] * kb + b) * 16 + 8 * h);
                dm[ct] = cq_h2f(dmins[cols[ct] * kb + b]);
                const uint32_t u[4] = {__builtin_amdgcn_perm(w.x, w.x, 0x0c010c00u) | 0x64006400u, __builtin_amdgcn_perm(w.x, w.x, 0x0c030c02u) | 0x64006400u,
                                       __builtin_amdgcn_perm(w.y, w.y, 0x0c010c00u) | 0x64006400u, __builtin_amdgcn_perm(w.y, w.y, 0x0c030c02u) | 0x64006400u};
                mv[ct] = __builtin_bit_cast(v8h, u);   // 0x6400 | v is the f16 1024 + v
#pragma unroll
                for (int i = 0; i < 8; i++) mv[ct][i] -= k1024;
            }
#pragma unroll
            for (int rt = 0; rt < RT; rt++) sv[rt] = *(const v8h *)(a.bsh + ((b * a.m_stride + r0 + 32 * rt + (lane & 31)) * 16 + 8 * h));
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
                float dr[16];
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const float4 f = *(const float4 *)(a.dT + b * a.m_stride + r0 + 32 * rt + 8 * g + 4 * h);
                    dr[4 * g] = f.x, dr[4 * g + 1] = f.y, dr[4 * g + 2] = f.z, dr[4 * g + 3] = f.w;
                }
#pragma unroll
                for (int ct = 0; ct < CT; ct++) {
                    const v16f s = __builtin_amdgcn_mfma_f32_32x32x16_f16(sv[rt], mv[ct], zero, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[rt][ct][i] += (dr[i] * dm[ct]) * s[i];
                }
            }
        }
    }
    add_tiles<SHARE, true, RT, CT>(acc, r0, c0, m, n, y);
}

// Few rows (decode, small batches): sixteen lanes per weight row, each one block out of sixteen at a time; lane 0 of the
// sixteen adds the block terms in order (the same terms, the same order as above).  Sixteen weight rows and four
// activation rows per workgroup, so that a launch has many workgroups where the kernel above would have few.
__global__ void __launch_bounds__(256) min16_small_kernel(const uint8_t *__restrict__ mins, const uint16_t *__restrict__ dmins,
                                                          cq_act_view a, int64_t n, int64_t kb, int64_t m, float *__restrict__ y) {
    __shared__ float part[kSmallRows][16][17];
    const int j = threadIdx.x & 15, cl = threadIdx.x >> 4;
    const int64_t c = (int64_t)blockIdx.x * 16 + cl;
    const int64_t cc = c < n ? c : n - 1, r0 = (int64_t)blockIdx.y * kSmallRows;
    float acc[kSmallRows] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int64_t sb = 0; sb < kb; sb += 16) {
        const int64_t b = sb + j;
        if (b < kb) {
            const uint4 mw = *(const uint4 *)(mins + (cc * kb + b) * 16);
            const float dmin = cq_h2f(dmins[cc * kb + b]);
            const uint32_t w[4] = {mw.x, mw.y, mw.z, mw.w};
#pragma unroll
            for (int r = 0; r < kSmallRows; r++) {
                float term = 0.0f;
                if (r0 + r < m) {
                    const int16_t *bs = a.bsums + ((r0 + r) * kb + b) * 16;
                    int summs = 0;
#pragma unroll
                    for (int g = 0; g < 16; g++) summs += (int)bs[g] * (int)((w[g >> 2] >> (8 * (g & 3))) & 0xff);
                    term = (a.d[(r0 + r) * kb + b] * dmin) * (float)summs;
                }
                part[r][cl][j] = term;
            }
        }
        __syncthreads();
        if (j == 0) {
            for (int jj = 0; jj < 16 && sb + jj < kb; jj++)
#pragma unroll
                for (int r = 0; r < kSmallRows; r++) acc[r] += part[r][cl][jj];
        }
        __syncthreads();
    }
    if (j == 0 && c < n)
        for (int r = 0; r < kSmallRows && r0 + r < m; r++) y[(r0 + r) * n + c] -= acc[r];
}

}  // namespace

// `apart`: a row's bits may not depend on how many rows there are.  For that, one kernel takes all of them (Q2K: its unshared tiles add
// the blocks in the small kernel's order, with the same roundings).
// Whether a tile of 64 x 64 for every wave would be fewer than one wave for each SIMD.
static bool share_tile(const cq_weight *w, int64_t m) { return m <= 32 || ((w->n + 63) / 64) * ((m + 63) / 64) < 4 * cq_num_cus(); }

hipError_t cq_launch_min32_term(const cq_weight *w, cq_act_view a, int64_t m, float *y, bool apart, hipStream_t s) {
    if (!cq_has_min32(w->ggml_dtype)) return hipErrorInvalidValue;
    if (m == 0 || w->n == 0 || w->k == 0) return hipSuccess;
    const int64_t nb = w->k / 32;
    const uint16_t *mins = (const uint16_t *)w->p2;
    if (apart)
        CQ_LAUNCH(min32_small_kernel, dim3((unsigned)((w->n + 15) / 16), (unsigned)((m + kSmallRows - 1) / kSmallRows)), 256, 0, s, mins, a,
                  w->n, nb, m, y);
    else if (share_tile(w, m))
        CQ_LAUNCH(min32_mfma_kernel<true>, dim3((unsigned)((w->n + 31) / 32), (unsigned)((m + 31) / 32)), 256, 0, s, mins, a, w->n, nb, m, y);
    else CQ_LAUNCH(min32_mfma_kernel<false>, dim3((unsigned)((w->n + 255) / 256), (unsigned)((m + 63) / 64)), 256, 0, s, mins, a, w->n, nb, m, y);
    return hipGetLastError();
}

hipError_t cq_launch_min16_term(const cq_weight *w, cq_act_view a, int64_t m, float *y, bool apart, hipStream_t s) {
    if (!cq_has_min16(w->ggml_dtype)) return hipErrorInvalidValue;
    if (m == 0 || w->n == 0 || w->k == 0) return hipSuccess;
    const uint16_t *dmins = (const uint16_t *)w->p5;
    const int64_t kb = w->k / 256;
    if (m <= kSmallRows)
        CQ_LAUNCH(min16_small_kernel, dim3((unsigned)((w->n + 15) / 16), (unsigned)((m + kSmallRows - 1) / kSmallRows)), 256, 0, s, w->p4,
                  dmins, a, w->n, kb, m, y);
    else if (!apart && share_tile(w, m))
        CQ_LAUNCH(min16_mfma_kernel<true>, dim3((unsigned)((w->n + 31) / 32), (unsigned)((m + 31) / 32)), 256, 0, s, w->p4, dmins, a, w->n, kb, m, y);
    else CQ_LAUNCH(min16_mfma_kernel<false>, dim3((unsigned)((w->n + 255) / 256), (unsigned)((m + 63) / 64)), 256, 0, s, w->p4, dmins, a, w->n, kb, m, y);
    return hipGetLastError();
}
