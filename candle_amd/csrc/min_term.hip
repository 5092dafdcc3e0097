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
// Many tiles: every wave one of 32 rows x 64 weight rows.  Few tiles: 32 x 32, their steps dealt to the four waves of a workgroup, since few rows
// leave too few tiles to fill the machine and one wave would walk the whole row by itself.
// Bound: the pass over y and the gather of the operands, 16 bytes of a row at a time.  Against the sums on the vector units through LDS, us a
// whole call before and after: Q5_1 2225 x 3328 with 3343 rows 187 -> 119, Q4_1 14336 x 4096 with 512 rows 184 -> 119, 4096 x 4096 with 64 rows
// 36.0 -> 21.0, Q2K 4096 x 4096 with 1024 rows 147 -> 81, with 128 rows 59.9 -> 28.7, 10400 x 768 with 561 rows 59 -> 36 (without the term:
// 94, 95, -, 58, -, 25).  A wave's part of y is requested before its sums are done: 10400 x 768 45.5 -> 36.2
// (few rows: the split-K kernels add the terms themselves, skinny.hip).  Error of the m * s term against 64 bits (4096 x 4096, 64 rows, relative
// rms): 8.9e-8 -> 6.0e-8.
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

// One column tile of y, requested ahead of the sums that are added to it (element i: row 8 * (i / 4) + 4 * (lane / 32) + i % 4).
__device__ __forceinline__ void load_tile(const float *y, int64_t r0, int64_t c, int64_t m, int64_t n, int h, v16f &old) {
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int64_t r = r0 + 8 * (i >> 2) + 4 * h + (i & 3);
        old[i] = r < m && c < n ? y[r * n + c] : 0.0f;
    }
}
// Adds (SUB: subtracts) the tiles.
template <bool SUB, int CT>
__device__ __forceinline__ void add_tiles(const v16f (&acc)[CT], const v16f (&old)[CT], int64_t r0, int64_t c0, int64_t m, int64_t n, float *y) {
    const int lane = threadIdx.x & 63, h = lane >> 5;
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        const int64_t c = c0 + 32 * ct + (lane & 31);
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int64_t r = r0 + 8 * (i >> 2) + 4 * h + (i & 3);
            if (r < m && c < n) y[r * n + c] = old[ct][i] + (SUB ? -acc[ct][i] : acc[ct][i]);
        }
    }
}
// The same for a tile whose four waves hold parts of the sums: added in order first.
template <bool SUB>
__device__ __forceinline__ void add_shared_tile(const v16f &acc, int64_t r0, int64_t c0, int64_t m, int64_t n, float *__restrict__ y) {
    __shared__ float part[4][16][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, h = lane >> 5;
    const int64_t c = c0 + (lane & 31), r = r0 + 8 * wave + 4 * h;   // wave w finishes result registers 4w .. 4w + 3
    float old[4];
#pragma unroll
    for (int j = 0; j < 4; j++) old[j] = r + j < m && c < n ? y[(r + j) * n + c] : 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i++) part[wave][i][lane] = acc[i];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int i = 4 * wave + j;
        const float t = ((part[0][i][lane] + part[1][i][lane]) + part[2][i][lane]) + part[3][i][lane];
        if (r + j < m && c < n) y[(r + j) * n + c] = old[j] + (SUB ? -t : t);
    }
}

__device__ __forceinline__ void load_scales(const float *row, int64_t b, int64_t nb, float (&d)[8]) {
    if (b + 8 <= nb) {
#pragma unroll
        for (int i = 0; i < 8; i++) d[i] = row[b + i];
    } else {
#pragma unroll
        for (int i = 0; i < 8; i++) d[i] = b + i < nb ? row[b + i] : 0.0f;
    }
}
// The s fields of eight blocks.
__device__ __forceinline__ v8h scaled_sums(const HalfRow &sums, const float (&d)[8]) {
    v8h s;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float hs = (float)(_Float16)(float)(int16_t)(sums.w[i >> 1] >> (16 * (i & 1)));
        s[i] = (_Float16)(hs * d[i]);
    }
    return s;
}
struct Raw32 {
    HalfRow mins, sums;
    float d[8];
};
__device__ __forceinline__ void load_raw32(const uint16_t *mins, const cq_act_view &a, int64_t col, int64_t row, int64_t b, int64_t nb, Raw32 &o) {
    o.mins = load_eight(mins, col, b, nb);
    o.sums = load_eight(a.bsum32, row, b, nb);
    load_scales(a.d + row * nb, b, nb, o.d);
}

// The steps of a 32 x 32 tile dealt to the waves.
__global__ void __launch_bounds__(256) min32_shared_kernel(const uint16_t *__restrict__ mins, cq_act_view a, int64_t n, int64_t nb, int64_t m, float *y) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, h = lane >> 5;
    const int64_t r0 = (int64_t)blockIdx.y * 32, c0 = (int64_t)blockIdx.x * 32;
    // (rows and weight rows past the end repeat the last one; their results are not stored)
    const int64_t row = r0 + (lane & 31) < m ? r0 + (lane & 31) : m - 1, col = c0 + (lane & 31) < n ? c0 + (lane & 31) : n - 1;
    v16f acc;
#pragma unroll
    for (int i = 0; i < 16; i++) acc[i] = 0.0f;
    Raw32 cur, nxt;
    int64_t b0 = 16 * wave;
    if (b0 < nb) load_raw32(mins, a, col, row, b0 + 8 * h, nb, cur);
    for (; b0 < nb; b0 += 64) {
        if (b0 + 64 < nb) load_raw32(mins, a, col, row, b0 + 64 + 8 * h, nb, nxt);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(scaled_sums(cur.sums, cur.d), __builtin_bit_cast(v8h, cur.mins), acc, 0, 0, 0);
        cur = nxt;
    }
    add_shared_tile<false>(acc, r0, c0, m, n, y);
}
// Every wave a 32 x 64 tile, the workgroup's four side by side.  The rows' s values are formed once a workgroup, 64 blocks at a time, in LDS; the
// minima of a weight row are read four steps at once, a whole line.  (Step by step a wave takes 32 bytes of every line it touches and the
// line is gone before the next step: four times the traffic from L2, 38 us of the 134 at 14336 x 4096 with 512 rows.)
__global__ void __launch_bounds__(256) min32_tiles_kernel(const uint16_t *__restrict__ mins, cq_act_view a, int64_t n, int64_t nb, int64_t m, float *y) {
    constexpr int CT = 2, kAhead = 64, kRow = kAhead + 8;   // (rows of 144 bytes: 16-byte reads of 32 rows meet every bank equally often)
    __shared__ __align__(16) _Float16 sv[32 * kRow];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, h = lane >> 5;
    const int64_t r0 = (int64_t)blockIdx.y * 32, c0 = ((int64_t)blockIdx.x * 4 + wave) * 32 * CT;
    const int srow = threadIdx.x >> 3, sblk = (threadIdx.x & 7) * 8;   // the s values this thread forms
    const int64_t row = r0 + srow < m ? r0 + srow : m - 1;
    v16f acc[CT], old[CT];
    int64_t cols[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        cols[ct] = c0 + 32 * ct + (lane & 31) < n ? c0 + 32 * ct + (lane & 31) : n - 1;
#pragma unroll
        for (int i = 0; i < 16; i++) acc[ct][i] = 0.0f;
    }
    for (int64_t b0 = 0; b0 < nb; b0 += kAhead) {
        HalfRow mw[4][CT];
#pragma unroll
        for (int ct = 0; ct < CT; ct++)
#pragma unroll
            for (int s = 0; s < 4; s++) mw[s][ct] = load_eight(mins, cols[ct], b0 + 16 * s + 8 * h, nb);
        float d[8];
        const HalfRow sums = load_eight(a.bsum32, row, b0 + sblk, nb);
        load_scales(a.d + row * nb, b0 + sblk, nb, d);
        if (b0 + kAhead >= nb) {   // (behind the last operands)
#pragma unroll
            for (int ct = 0; ct < CT; ct++) load_tile(y, r0, c0 + 32 * ct + (lane & 31), m, n, h, old[ct]);
        }
        if (b0) __syncthreads();   // the values of the blocks before have been read
        *(v8h *)(sv + srow * kRow + sblk) = scaled_sums(sums, d);
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 4; s++) {   // (blocks past the end: both factors zero)
            const v8h op = *(const v8h *)(sv + (lane & 31) * kRow + 16 * s + 8 * h);
#pragma unroll
            for (int ct = 0; ct < CT; ct++) acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_f16(op, __builtin_bit_cast(v8h, mw[s][ct]), acc[ct], 0, 0, 0);
        }
    }
    add_tiles<false, CT>(acc, old, r0, c0, m, n, y);
}

// ---- rows that keep their bits whatever the row count ----
// Two kernels with one order of the f32 additions: the blocks of a weight row in chunks of eight, a chunk's products added one after the
// other from zero, the chunk sums added one after the other.  (apart32_small says which takes a call.)
constexpr int kChunk = 8;

// A workgroup forms a 32 x 32 tile of outputs, thread (i, j) the 2 x 2 outputs (i, i+16) x (j, j+16); the minima and the s values of 32
// blocks at a time go through LDS.
constexpr int kT = 32, kB = 32;
__global__ void __launch_bounds__(256) min32_tile_kernel(const uint16_t *__restrict__ mins, cq_act_view a, int64_t n, int64_t nb,
                                                         int64_t m, float *__restrict__ y) {
    __shared__ float sm[kT][kB + 1], ss[kT][kB + 1];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int64_t c0 = (int64_t)blockIdx.x * kT, r0 = (int64_t)blockIdx.y * kT;
    float acc[2][2] = {{0.0f, 0.0f}, {0.0f, 0.0f}};
    for (int64_t b0 = 0; b0 < nb; b0 += kB) {
        for (int e = threadIdx.x; e < kT * kB; e += 256) {
            const int row = e / kB, bb = e % kB;
            const int64_t b = b0 + bb;
            const bool ok = b < nb;
            sm[row][bb] = ok && c0 + row < n ? cq_h2f(mins[(c0 + row) * nb + b]) : 0.0f;
            ss[row][bb] = ok && r0 + row < m ? block_s(a, (r0 + row) * nb + b) : 0.0f;
        }
        __syncthreads();
        for (int g = 0; g < kB && b0 + g < nb; g += kChunk) {
            float t[2][2] = {{0.0f, 0.0f}, {0.0f, 0.0f}};
#pragma unroll
            for (int i = 0; i < kChunk; i++) {
                if (b0 + g + i < nb) {   // blocks past the end of the row are left out, not added as zeros
                    const float s0 = ss[ty][g + i], s1 = ss[ty + 16][g + i], m0 = sm[tx][g + i], m1 = sm[tx + 16][g + i];
                    t[0][0] += m0 * s0;
                    t[0][1] += m1 * s0;
                    t[1][0] += m0 * s1;
                    t[1][1] += m1 * s1;
                }
            }
            acc[0][0] += t[0][0];
            acc[0][1] += t[0][1];
            acc[1][0] += t[1][0];
            acc[1][1] += t[1][1];
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int64_t r = r0 + ty + 16 * i, c = c0 + tx + 16 * j;
            if (r < m && c < n) y[r * n + c] += acc[i][j];
        }
}

// Few outputs: sixteen lanes per weight row, each a chunk of eight blocks out of 128 at a time; lane
// 0 of the sixteen adds the chunk sums in order.  Sixteen weight rows and four activation rows per workgroup.
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
template <int CT> struct Raw16 {
    uint2 mins[CT];
    uint16_t dmin[CT];
    v8h sums;
    float4 d[4];
};
template <int CT>
__device__ __forceinline__ void load_raw16(const uint8_t *mins, const uint16_t *dmins, const cq_act_view &a, const int64_t (&cols)[CT], int64_t r0,
                                           int64_t b, int64_t kb, int lane, Raw16<CT> &o) {
    const int h = lane >> 5;
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        o.mins[ct] = *(const uint2 *)(mins + (cols[ct] * kb + b) * 16 + 8 * h);
        o.dmin[ct] = dmins[cols[ct] * kb + b];
    }
    o.sums = *(const v8h *)(a.bsh + ((b * a.m_stride + r0 + (lane & 31)) * 16 + 8 * h));
#pragma unroll
    for (int g = 0; g < 4; g++) o.d[g] = *(const float4 *)(a.dT + b * a.m_stride + r0 + 8 * g + 4 * h);
}
template <bool SHARE>
__global__ void __launch_bounds__(256) min16_mfma_kernel(const uint8_t *__restrict__ mins, const uint16_t *__restrict__ dmins, cq_act_view a,
                                                         int64_t n, int64_t kb, int64_t m, float *y) {
    constexpr int CT = SHARE ? 1 : 2;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, h = lane >> 5;
    const int64_t r0 = (int64_t)blockIdx.y * 32, c0 = ((int64_t)blockIdx.x * (SHARE ? 1 : 4) + (SHARE ? 0 : wave)) * 32 * CT;
    v16f acc[CT], old[CT], zero;
    int64_t cols[CT];   // (weight rows past the end repeat the last one; rows past the end are the workspace's padding; neither is stored)
#pragma unroll
    for (int i = 0; i < 16; i++) zero[i] = 0.0f;
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        cols[ct] = c0 + 32 * ct + (lane & 31) < n ? c0 + 32 * ct + (lane & 31) : n - 1;
        acc[ct] = zero;
    }
    if (SHARE || c0 < n) {
        const int64_t step = SHARE ? 4 : 1;
        Raw16<CT> cur, nxt;
        int64_t b = SHARE ? wave : 0;
        if (b < kb) load_raw16<CT>(mins, dmins, a, cols, r0, b, kb, lane, cur);
        if constexpr (!SHARE) {
#pragma unroll
            for (int ct = 0; ct < CT; ct++) load_tile(y, r0, c0 + 32 * ct + (lane & 31), m, n, h, old[ct]);
        }
        for (; b < kb; b += step) {
            if (b + step < kb) load_raw16<CT>(mins, dmins, a, cols, r0, b + step, kb, lane, nxt);
#pragma unroll
            for (int ct = 0; ct < CT; ct++) {
                const uint2 w = cur.mins[ct];
                const uint32_t u[4] = {__builtin_amdgcn_perm(w.x, w.x, 0x0c010c00u) | 0x64006400u, __builtin_amdgcn_perm(w.x, w.x, 0x0c030c02u) | 0x64006400u,
                                       __builtin_amdgcn_perm(w.y, w.y, 0x0c010c00u) | 0x64006400u, __builtin_amdgcn_perm(w.y, w.y, 0x0c030c02u) | 0x64006400u};
                v8h mv = __builtin_bit_cast(v8h, u);   // 0x6400 | v is the f16 1024 + v
#pragma unroll
                for (int i = 0; i < 8; i++) mv[i] -= (_Float16)1024.0f;
                const float dm = cq_h2f(cur.dmin[ct]);
                const v16f s = __builtin_amdgcn_mfma_f32_32x32x16_f16(cur.sums, mv, zero, 0, 0, 0);
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const float dr[4] = {cur.d[g].x, cur.d[g].y, cur.d[g].z, cur.d[g].w};
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[ct][4 * g + i] += (dr[i] * dm) * s[4 * g + i];
                }
            }
            cur = nxt;
        }
    }
    if constexpr (SHARE) add_shared_tile<true>(acc[0], r0, c0, m, n, y);
    else if (c0 < n) add_tiles<true, CT>(acc, old, r0, c0, m, n, y);
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

// Whether a tile for every wave would be fewer than one wave for each SIMD.
static bool share_tile(const cq_weight *w, int64_t m) { return ((w->n + 63) / 64) * ((m + 31) / 32) < 4 * cq_num_cus(); }

// A workgroup names its rows by blockIdx.y, a grid has 65535 of those at most: more rows than the smallest groups make of them go in
// several launches (a whole number of four rows each: the scales of the tiles are read four rows at a time).
constexpr int64_t kMostRows = (int64_t)65535 * kSmallRows;

// `apart`: a row's bits may not depend on how many rows there are: the kernels with one order of the sums.  The one of sixteen lanes a weight
// row up to four rows, and for rows of 80 blocks and more (fewer leave most of a chunk's lanes idle) up to 24000 outputs.  Whole calls, us,
// 32 x 32 tiles / sixteen lanes: Q4_1 with 8 rows 4096 x 128 13.8 / 16.4, 4096 x 4096 28.5 / 30.0, 300 x 4096 26.7 / 23.0, with 16 rows 1000 x
// 2560 32.0 / 30.3, 300 x 2048 28.2 / 28.4, with 64 rows 4096 x 4096 112 / 191, 300 x 4096 97.8 / 97.1, 8 x 4096 94.3 / 87.7.
static bool apart32_small(const cq_weight *w, int64_t m) { return m <= kSmallRows || (w->k >= 80 * 32 && w->n * m <= 24000); }
// Q2K: the tiles without sharing add the blocks in the small kernel's order, with the same roundings.  Up to 64 rows the small kernel, but for many
// outputs of short rows.  Whole calls, us, tiles / small: 8 rows 8 x 4096 26.0 / 19.1, 5 rows 4096 x 1280 21.6 / 19.3, 64 rows 4096 x 4096
// 129 / 127, 4096 x 1280 114.6 / 117.4, 4096 x 256 99.8 / 104.9.
static bool apart16_small(const cq_weight *w, int64_t m) { return m <= 64 && (w->k > 8 * QK_K || w->n * m <= (1 << 17)); }

static void launch_min32(const cq_weight *w, const cq_act_view &a, int64_t m, float *y, bool apart, hipStream_t s) {
    const int64_t nb = w->k / 32;
    const uint16_t *mins = (const uint16_t *)w->p2;
    if (apart && apart32_small(w, m))
        CQ_LAUNCH(min32_small_kernel, dim3((unsigned)((w->n + 15) / 16), (unsigned)((m + kSmallRows - 1) / kSmallRows)), 256, 0, s, mins, a,
                  w->n, nb, m, y);
    else if (apart) CQ_LAUNCH(min32_tile_kernel, dim3((unsigned)((w->n + kT - 1) / kT), (unsigned)((m + kT - 1) / kT)), 256, 0, s, mins, a, w->n, nb, m, y);
    else if (share_tile(w, m))
        CQ_LAUNCH(min32_shared_kernel, dim3((unsigned)((w->n + 31) / 32), (unsigned)((m + 31) / 32)), 256, 0, s, mins, a, w->n, nb, m, y);
    else CQ_LAUNCH(min32_tiles_kernel, dim3((unsigned)((w->n + 255) / 256), (unsigned)((m + 31) / 32)), 256, 0, s, mins, a, w->n, nb, m, y);
}
hipError_t cq_launch_min32_term(const cq_weight *w, cq_act_view a, int64_t m, float *y, bool apart, hipStream_t s) {
    if (!cq_has_min32(w->ggml_dtype)) return hipErrorInvalidValue;
    if (m == 0 || w->n == 0 || w->k == 0) return hipSuccess;
    for (int64_t r = 0; r < m; r += kMostRows) {
        cq_act_view v = a;
        v.d += r * (w->k / 32);
        v.bsum32 += r * (w->k / 32);
        launch_min32(w, v, m - r < kMostRows ? m - r : kMostRows, y + r * w->n, apart, s);
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    }
    return hipSuccess;
}

static void launch_min16(const cq_weight *w, const cq_act_view &a, int64_t m, float *y, bool apart, hipStream_t s) {
    const uint16_t *dmins = (const uint16_t *)w->p5;
    const int64_t kb = w->k / 256;
    if (m <= kSmallRows || (apart && apart16_small(w, m)))
        CQ_LAUNCH(min16_small_kernel, dim3((unsigned)((w->n + 15) / 16), (unsigned)((m + kSmallRows - 1) / kSmallRows)), 256, 0, s, w->p4,
                  dmins, a, w->n, kb, m, y);
    else if (!apart && share_tile(w, m))
        CQ_LAUNCH(min16_mfma_kernel<true>, dim3((unsigned)((w->n + 31) / 32), (unsigned)((m + 31) / 32)), 256, 0, s, w->p4, dmins, a, w->n, kb, m, y);
    else CQ_LAUNCH(min16_mfma_kernel<false>, dim3((unsigned)((w->n + 255) / 256), (unsigned)((m + 31) / 32)), 256, 0, s, w->p4, dmins, a, w->n, kb, m, y);
}
hipError_t cq_launch_min16_term(const cq_weight *w, cq_act_view a, int64_t m, float *y, bool apart, hipStream_t s) {
    if (!cq_has_min16(w->ggml_dtype)) return hipErrorInvalidValue;
    if (m == 0 || w->n == 0 || w->k == 0) return hipSuccess;
    for (int64_t r = 0; r < m; r += kMostRows) {
        cq_act_view v = a;   // (row-major planes by row, block-major ones by place)
        v.d += r * (w->k / 256);
        v.bsums += r * (w->k / 256) * 16;
        v.dT += r;
        v.bsh += r * 16;
        launch_min16(w, v, m - r < kMostRows ? m - r : kMostRows, y + r * w->n, apart, s);
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    }
    return hipSuccess;
}
