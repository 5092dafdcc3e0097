// Weight quantizers on the device: f32 -> GGML blocks (array-of-blocks bytes), the
// arithmetic of T::from_float in candle-core/src/quantized/k_quants.rs and utils.rs,
// every f32 operation a single IEEE operation in the reference's order (compiled with
// -ffp-contract=off).  The reference's CUDA arm copies the tensor to the host and quantizes
// there (cuda.rs:448-472); the bytes produced here are the same.
//   Q4_0 k_quants.rs:185-220      Q8_0 :586-615
//   Q4K  :1252-1311 + utils.rs:201-258 (make_qkx1_quants) + :49-59 (get_scale_min_k4)
//   Q5K  :1450-1525, the same with 32 levels
//   Q6K  :1643-1713 + utils.rs:61-198  (make_qx_quants, n=16, nmax=32, rmse_type=1)
//   Q2K  :770-839 (make_qkx1_quants over 16 elements, 3 levels)
//   Q4_1 :296-326   Q5_1 :496-530   Q5_0 :393-425   Q3K  :1011-1090 + utils.rs:261-326 (make_q3_quants, nmax=4, do_rmse)
//
// Bound: vector instructions (the scale searches run over a group five times, their sums one element after the other
// as the reference adds them).  So the unit of work is a lane per scale group (32 or 16 elements), its elements and
// quants in registers: eight or sixteen times the lanes of one lane per 256-element block, and no array in scratch.
// A workgroup's elements come in through LDS in whole lines (rows padded by four floats, so that the lanes' 16-byte
// reads of their own groups spread over the banks); what the groups of a block share (scales, quants that meet in one
// byte) goes through LDS too, where the finished blocks are put together and then stored straight to the weight's planes.
// 11008 x 4096 elements (180 MB read), a lane per block before -> now: Q4K / Q5K 1730 / 1704 -> 119 / 121 us, Q2K 1105 -> 129,
// Q3K 1574 -> 183, Q6K 520 -> 201, Q4_0 75 -> 36, Q4_1 97 -> 37, Q5_0 171 -> 40, Q5_1 174 -> 40, Q8_0 163 -> 42 (4.9-5.4 TB/s).
// Without GGML blocks in memory between the quantizer and the planes (no temporary to allocate, 12-15 us less of re-packing), a whole
// call that creates and quantizes 11008 x 4096: Q4K 215 -> 182 us, Q4_0 127 -> 94, Q6K 530 -> 261, Q8_0 383 -> 97, Q5_1 430 -> 113.
#include "repack_units.h"

namespace {

constexpr int kLanes = 256;   // lanes (= groups) of a workgroup

typedef float f4_any __attribute__((ext_vector_type(4), aligned(4)));   // src may be any contiguous f32 view

// The workgroup's kLanes groups of G floats, each lane its own (past the last group: the last one again).
template <int G> __device__ __forceinline__ void load_groups(const float *__restrict__ src, int64_t ngroups, float *lds, float (&x)[G]) {
    constexpr int V = G / 4, RS = G + 4;
    const int64_t g0 = (int64_t)blockIdx.x * kLanes;
#pragma unroll
    for (int i = 0; i < V; i++) {
        const int idx = i * kLanes + (int)threadIdx.x, grp = idx / V, c = idx % V;
        const int64_t g = g0 + grp < ngroups ? g0 + grp : ngroups - 1;
        const f4_any v = __builtin_nontemporal_load((const f4_any *)(src + g * G + c * 4));
        *(float4 *)(lds + grp * RS + c * 4) = make_float4(v.x, v.y, v.z, v.w);
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < V; c++) {
        const float4 v = *(const float4 *)(lds + (int)threadIdx.x * RS + c * 4);
        x[4 * c] = v.x; x[4 * c + 1] = v.y; x[4 * c + 2] = v.z; x[4 * c + 3] = v.w;
    }
    __syncthreads();   // the same LDS takes the finished blocks
}

// The workgroup's blocks from their LDS image to the weight's planes, PER of them in a full workgroup.
template <int DT, int PER> __device__ __forceinline__ void store_blocks(uint8_t *img, int64_t nblocks, const cq_planes &pl) {
    constexpr int U = Ggml<DT>::kUnits;
    const int64_t b0 = (int64_t)blockIdx.x * PER;
    const int count = (int)(nblocks - b0 < PER ? nblocks - b0 : PER);
    __syncthreads();
    for (int i = threadIdx.x; i < count * U; i += kLanes) repack_unit<DT, false>(img + i / U * Ggml<DT>::kSize, b0 + i / U, i % U, pl);
}

__device__ __forceinline__ void put16(uint8_t *p, uint16_t v) { *(uint16_t *)p = v; }   // (blocks lie at even offsets)
template <int N> __device__ __forceinline__ void put_bytes(uint8_t *p, const uint32_t (&w)[N]) {
#pragma unroll
    for (int i = 0; i < N; i++) {
        put16(p + 4 * i, (uint16_t)w[i]);
        put16(p + 4 * i + 2, (uint16_t)(w[i] >> 16));
    }
}

// clamp(nearest_int(v), 0, top) for top <= 130: with the clamp in front, rounding is one conversion (cq_round_away_i32);
// NaN gives 0 as in nearest_int.
__device__ __forceinline__ int round_unsigned(float v, float top) {
    int r;
    asm("v_cvt_rpi_i32_f32_e32 %0, %1" : "=v"(r) : "v"(fminf(fmaxf(v, 0.0f), top)));
    return r;
}
// clamp(nearest_int(v), lo, hi) for |lo|, |hi| <= 128: magnitude clamped (NaN to 0) and rounded, the sign put back.
__device__ __forceinline__ int round_signed(float v, int lo, int hi) {
    const int m = round_unsigned(fabsf(v), 130.0f), sgn = __builtin_bit_cast(int, v) >> 31;
    return cq_clampi((m ^ sgn) - sgn, lo, hi);
}

// ---------------------------------------------------------------------- blocks of 32: a lane per block ----
template <int DT>
__global__ void __launch_bounds__(kLanes) quantize_blk32(const float *__restrict__ src, int64_t nblocks, cq_planes pl) {
    constexpr int TS = Ggml<DT>::kSize;
    __shared__ __align__(16) float lds[kLanes * 36];
    float x[32];
    load_groups<32>(src, nblocks, lds, x);
    uint8_t *img = (uint8_t *)lds, *y = img + (int)threadIdx.x * TS;
    if constexpr (DT == CQ_DTYPE_Q8_0) {
        float amax = 0.0f;
#pragma unroll
        for (int j = 0; j < 32; j++) amax = fmaxf(amax, fabsf(x[j]));
        const float d = amax / 127.0f;
        const float id = d != 0.0f ? 1.0f / d : 0.0f;
        put16(y, cq_f2h(d));
        uint32_t w[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            w[i] = 0;
#pragma unroll
            for (int c = 0; c < 4; c++) w[i] |= (uint32_t)(uint8_t)cq_as_i8(roundf(x[4 * i + c] * id)) << (8 * c);
        }
        put_bytes(y + 2, w);
    } else if constexpr (DT == CQ_DTYPE_Q4_0 || DT == CQ_DTYPE_Q5_0) {
        constexpr bool FIVE = DT == CQ_DTYPE_Q5_0;
        float amax = 0.0f, max = 0.0f;
#pragma unroll
        for (int j = 0; j < 32; j++)
            if (amax < fabsf(x[j])) { amax = fabsf(x[j]); max = x[j]; }
        const float d = max / (FIVE ? -16.0f : -8.0f);
        const float id = d != 0.0f ? 1.0f / d : 0.0f;
        put16(y, cq_f2h(d));
        uint32_t w[4] = {0, 0, 0, 0}, qh = 0;
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const float x0 = x[j] * id, x1 = x[16 + j] * id;
            uint32_t xi0, xi1;
            if (FIVE) {
                const int8_t s0 = cq_as_i8(x0 + 16.5f), s1 = cq_as_i8(x1 + 16.5f);
                xi0 = (uint8_t)(s0 < 31 ? s0 : 31);
                xi1 = (uint8_t)(s1 < 31 ? s1 : 31);
                qh |= ((xi0 >> 4) & 1u) << j;
                qh |= ((xi1 >> 4) & 1u) << (j + 16);
            } else {
                xi0 = cq_as_u8(x0 + 8.5f);
                xi1 = cq_as_u8(x1 + 8.5f);
                if (xi0 > 15) xi0 = 15;
                if (xi1 > 15) xi1 = 15;
            }
            w[j >> 2] |= ((xi0 & 15u) | ((xi1 & 15u) << 4)) << (8 * (j & 3));
        }
        if (FIVE) {
            const uint32_t q[1] = {qh};
            put_bytes(y + 2, q);
        }
        put_bytes(y + (FIVE ? 6 : 2), w);
    } else {
        // Q4_1, Q5_1: d = (max - min) / levels, quants round((x - min) / d)
        constexpr bool FIVE = DT == CQ_DTYPE_Q5_1;
        float min = INFINITY, max = -INFINITY;
#pragma unroll
        for (int j = 0; j < 32; j++) {
            min = fminf(x[j], min);   // f32::min / f32::max: a NaN operand loses
            max = fmaxf(x[j], max);
        }
        const float d = (max - min) / (FIVE ? 31.0f : 15.0f);
        const float id = d != 0.0f ? 1.0f / d : 0.0f;
        put16(y, cq_f2h(d));
        put16(y + 2, cq_f2h(min));
        uint32_t w[4] = {0, 0, 0, 0}, qh = 0;
#pragma unroll
        for (int j = 0; j < 16; j++) {
            uint32_t xi0 = cq_as_u8((x[j] - min) * id + 0.5f), xi1 = cq_as_u8((x[16 + j] - min) * id + 0.5f);
            if (!FIVE) {
                if (xi0 > 15) xi0 = 15;
                if (xi1 > 15) xi1 = 15;
            }
            w[j >> 2] |= ((xi0 & 15u) | ((xi1 & 15u) << 4)) << (8 * (j & 3));
            qh |= ((xi0 >> 4) & 1u) << j;
            qh |= ((xi1 >> 4) & 1u) << (j + 16);
        }
        if (FIVE) {
            const uint32_t q[1] = {qh};
            put_bytes(y + 4, q);
        }
        put_bytes(y + (FIVE ? 8 : 4), w);
    }
    store_blocks<DT, kLanes>(img, nblocks, pl);
}

// ------------------------------------------------------------------- blocks of 256: a lane per group ----
// utils.rs:201-258
template <int N> __device__ __forceinline__ void make_qkx1_quants(const float (&x)[N], int nmax, float &out_scale, float &out_min) {
    const int ntry = 5;
    float min = x[0], max = x[0];
#pragma unroll
    for (int i = 1; i < N; i++) {
        if (x[i] < min) min = x[i];
        if (x[i] > max) max = x[i];
    }
    if (max == min) { out_scale = 0.0f; out_min = 0.0f; return; }
    float l[N];   // the quants of the last try
#pragma unroll
    for (int i = 0; i < N; i++) l[i] = 0.0f;
    min = fminf(min, 0.0f);
    const float top = (float)nmax;
    float iscale = top / (max - min);
    float scale = 1.0f / iscale;
    for (int t = 0; t < ntry; t++) {
        float sumlx = 0.0f;
        int32_t suml2 = 0;
        bool did_change = false;
#pragma unroll
        for (int i = 0; i < N; i++) {
            const float v = x[i] - min;
            const int li = round_unsigned(iscale * v, top);
            const float lf = (float)li;
            did_change = did_change || lf != l[i];
            l[i] = lf;
            sumlx += v * lf;
            suml2 += (int32_t)__umul24((uint32_t)li, (uint32_t)li);
        }
        scale = sumlx / (float)suml2;
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < N; i++) sum += x[i] - scale * l[i];
        min = sum / (float)N;
        if (min > 0.0f) min = 0.0f;
        iscale = 1.0f / scale;
        if (!did_change) break;
    }
    out_scale = scale;
    out_min = -min;
}

// Largest of the values of eight neighbouring lanes (the groups of one block), and zero.
__device__ __forceinline__ float max_of_8(float v) {
    v = fmaxf(v, dpp_f<kQuadSwap1>(v));
    v = fmaxf(v, dpp_f<kQuadSwap2>(v));
    v = fmaxf(v, dpp_f<kHalfMirror>(v));
    return fmaxf(v, 0.0f);
}

// LEVELS = 16: Q4K (144-byte blocks).  LEVELS = 32: Q5K (k_quants.rs:1450-1525), the same scale search
// with 31 as the top level, the quants' fifth bits in qh[32] between the scales and the nibbles.
template <int LEVELS>
__global__ void __launch_bounds__(kLanes) quantize_q4k(const float *__restrict__ src, int64_t nblocks, cq_planes pl) {
    constexpr int DT = LEVELS == 16 ? CQ_DTYPE_Q4K : CQ_DTYPE_Q5K, TS = Ggml<DT>::kSize, PER = kLanes / 8;
    constexpr int kQs = LEVELS == 16 ? 16 : 48;   // offset of the nibbles in the block
    __shared__ __align__(16) float lds[kLanes * 36];
    __shared__ __align__(16) uint8_t codes[kLanes * 2];   // per block: eight scale codes, eight min codes
    const int t = threadIdx.x, blk = t >> 3, j = t & 7;
    float x[32];
    load_groups<32>(src, nblocks * 8, lds, x);
    float scale, min;
    make_qkx1_quants<32>(x, LEVELS - 1, scale, min);
    const float max_scale = max_of_8(scale), max_min = max_of_8(min);
    const float inv_scale = max_scale > 0.0f ? 63.0f / max_scale : 0.0f;
    const float inv_min = max_min > 0.0f ? 63.0f / max_min : 0.0f;
    int32_t lsi = cq_nearest_int(inv_scale * scale), lmi = cq_nearest_int(inv_min * min);
    if (lsi > 63) lsi = 63;
    if (lmi > 63) lmi = 63;
    codes[blk * 16 + j] = (uint8_t)lsi;
    codes[blk * 16 + 8 + j] = (uint8_t)lmi;
    __syncthreads();
    const uint4 c = *(const uint4 *)(codes + blk * 16);   // scale codes 0..3, 4..7, min codes 0..3, 4..7
    const uint32_t u0 = c.x | ((c.y << 2) & 0xC0C0C0C0u), u1 = c.z | ((c.w << 2) & 0xC0C0C0C0u);
    const uint32_t u2 = (c.y & 0x0F0F0F0Fu) | ((c.w & 0x0F0F0F0Fu) << 4);
    const uint16_t dh = cq_f2h(max_scale / 63.0f), dminh = cq_f2h(max_min / 63.0f);
    int sc, m;
    cq_scale_min_k4(j, u0, u1, u2, sc, m);
    const float d = cq_h2f(dh) * (float)sc;
    uint32_t q[8];   // this group's 32 quants, one byte each
#pragma unroll
    for (int i = 0; i < 8; i++) q[i] = 0;
    if (d != 0.0f) {
        const float dm = cq_h2f(dminh) * (float)m;
#pragma unroll
        for (int i = 0; i < 32; i++) q[i >> 2] |= (uint32_t)round_unsigned((x[i] + dm) / d, (float)(LEVELS - 1)) << (8 * (i & 3));
    }
    uint8_t *img = (uint8_t *)lds, *y = img + blk * TS;
    // The groups 2g and 2g+1 (this lane and its neighbour) share 32 bytes, low and high nibbles: the even lane writes the
    // first sixteen bytes, the odd lane the others.
    const bool odd = j & 1;
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t mine = odd ? q[4 + i] : q[i], give = odd ? q[i] : q[4 + i];
        const uint32_t got = (uint32_t)dpp_i<kQuadSwap1>((int)give);
        const uint32_t lo = odd ? got : mine, hi = odd ? mine : got;
        w[i] = (lo & 0x0F0F0F0Fu) | ((hi & 0x0F0F0F0Fu) << 4);
        if (LEVELS == 32) q[i] = ((lo >> 4) & 0x01010101u) | (((hi >> 4) & 0x01010101u) << 1);   // fifth bits of the pair
    }
    *(uint4 *)(y + kQs + 16 * j) = make_uint4(w[0], w[1], w[2], w[3]);
    if (LEVELS == 32) {
        // qh[l]: bits 2g and 2g+1 from pair g; the four pairs of a block sit in lanes j = 0, 2, 4, 6 (odd: 1, 3, 5, 7)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t v = q[i] << (2 * (j >> 1));
            v |= (uint32_t)dpp_i<kQuadSwap2>((int)v);
            // the other four lanes in mirrored order hold the other parity: swap neighbours first
            const uint32_t s = (uint32_t)dpp_i<kQuadSwap1>((int)v);
            v |= (uint32_t)dpp_i<kHalfMirror>((int)s);
            w[i] = v;
        }
        if (j < 2) *(uint4 *)(y + 16 + 16 * j) = make_uint4(w[0], w[1], w[2], w[3]);
    }
    if (j == 0) *(uint4 *)y = make_uint4((uint32_t)dh | ((uint32_t)dminh << 16), u0, u1, u2);
    store_blocks<DT, PER>(img, nblocks, pl);
}

// utils.rs:61-198 specialised to n = 16, nmax = 32, rmse_type = 1 (weights w = x*x; returns after
// the five refinement passes, utils.rs:168-170).  ls: the quants, 0..63.
__device__ __forceinline__ float make_qx_quants_16_32(const float (&x)[16], int (&ls)[16]) {
    const int n = 16, nmax = 32;
    float max = 0.0f, amax = 0.0f;
#pragma unroll
    for (int i = 0; i < n; i++) {
        const float ax = fabsf(x[i]);
        if (ax > amax) { amax = ax; max = x[i]; }
    }
    if (amax == 0.0f) {
#pragma unroll
        for (int i = 0; i < n; i++) ls[i] = 0;
        return 0.0f;
    }
    const float iscale = -(float)nmax / max;
    float sumlx = 0.0f, suml2 = 0.0f;
#pragma unroll
    for (int i = 0; i < n; i++) {
        const int32_t l = round_signed(iscale * x[i], -nmax, nmax - 1);
        ls[i] = l + nmax;
        const float w = x[i] * x[i];
        const float lf = (float)l;
        sumlx += w * x[i] * lf;
        suml2 += w * lf * lf;
    }
    float scale = sumlx / suml2;
    float best = scale * sumlx;
    for (int itry = 0; itry < 3; itry++) {
        const float is2 = 1.0f / scale;
        float slx = 0.0f, sl2 = 0.0f;
        bool changed = false;
        int nl[16];
#pragma unroll
        for (int i = 0; i < n; i++) {
            const int32_t l = round_signed(is2 * x[i], -nmax, nmax - 1);
            nl[i] = l + nmax;
            changed = changed || nl[i] != ls[i];
            const float w = x[i] * x[i];
            const float lf = (float)l;
            slx += w * x[i] * lf;
            sl2 += w * lf * lf;
        }
        if (!changed || sl2 == 0.0f || slx * slx <= best * sl2) break;
#pragma unroll
        for (int i = 0; i < n; i++) ls[i] = nl[i];
        sumlx = slx;
        suml2 = sl2;
        scale = sumlx / suml2;
        best = scale * sumlx;
    }
    for (int itry = 0; itry < 5; itry++) {
        bool changed = false;
#pragma unroll
        for (int i = 0; i < n; i++) {
            const float w = x[i] * x[i];
            const int32_t l = ls[i] - nmax;
            float slx = sumlx - w * x[i] * (float)l;
            if (slx > 0.0f) {
                float sl2 = suml2 - w * (float)l * (float)l;
                const int32_t new_l = round_signed(x[i] * sl2 / slx, -nmax, nmax - 1);
                if (new_l != l) {
                    slx += w * x[i] * (float)new_l;
                    sl2 += w * (float)new_l * (float)new_l;
                    if (sl2 > 0.0f && slx * slx * suml2 > sumlx * sumlx * sl2) {
                        ls[i] = nmax + new_l;
                        sumlx = slx;
                        suml2 = sl2;
                        scale = sumlx / suml2;
                        changed = true;
                    }
                }
            }
        }
        if (!changed) break;
    }
    return scale;
}

// The sixteen scales of this lane's block, one per group, through LDS (`scales`: one float per lane of the workgroup).
__device__ __forceinline__ void share_scales(float *scales, float mine, float (&all)[16]) {
    scales[threadIdx.x] = mine;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float4 v = *(const float4 *)(scales + ((int)threadIdx.x & ~15) + 4 * i);
        all[4 * i] = v.x; all[4 * i + 1] = v.y; all[4 * i + 2] = v.z; all[4 * i + 3] = v.w;
    }
}

// Sixteen quants of a group as four words of bytes.
__device__ __forceinline__ uint4 pack16(const int (&q)[16]) {
    uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 16; i++) w[i >> 2] |= (uint32_t)q[i] << (8 * (i & 3));
    return make_uint4(w[0], w[1], w[2], w[3]);
}

__global__ void __launch_bounds__(kLanes) quantize_q6k(const float *__restrict__ src, int64_t nblocks, cq_planes pl) {
    constexpr int DT = CQ_DTYPE_Q6K, TS = Ggml<DT>::kSize, PER = kLanes / 16;
    __shared__ __align__(16) float lds[kLanes * 20];
    __shared__ __align__(16) float scales[kLanes];
    __shared__ __align__(16) uint4 quants[kLanes];
    const int t = threadIdx.x, blk = t >> 4, j = t & 15;
    float x[16], all[16];
    int l[16];
    load_groups<16>(src, nblocks * 16, lds, x);
    share_scales(scales, make_qx_quants_16_32(x, l), all);
    float max_scale = 0.0f, max_abs_scale = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const float a = fabsf(all[i]);
        if (a > max_abs_scale) { max_abs_scale = a; max_scale = all[i]; }
    }
    const float iscale = -128.0f / max_scale;
    const uint16_t dh = cq_f2h(1.0f / iscale);
    int32_t v = cq_nearest_int(iscale * scales[t]);
    if (v > 127) v = 127;
    const int8_t sc8 = (int8_t)v;
    const float d = cq_h2f(dh) * (float)sc8;
    if (d != 0.0f) {
#pragma unroll
        for (int i = 0; i < 16; i++) l[i] = round_signed(x[i] / d, -32, 31) + 32;
    }
    quants[t] = pack16(l);
    __syncthreads();
    uint8_t *img = (uint8_t *)lds, *y = img + blk * TS;
    const uint4 *Q = quants + blk * 16;
    y[192 + j] = (uint8_t)sc8;
    if (j < 8) {
        // ql bytes 16j ..: elements 128h + li (low nibbles) and 128h + li + 64 (high), li = 16 (j % 4) ..
        const int a = 8 * (j >> 2) + (j & 3);
        const uint4 lo = Q[a], hi = Q[a + 4];
        uint32_t w[4];
        w[0] = (lo.x & 0x0F0F0F0Fu) | ((hi.x & 0x0F0F0F0Fu) << 4);
        w[1] = (lo.y & 0x0F0F0F0Fu) | ((hi.y & 0x0F0F0F0Fu) << 4);
        w[2] = (lo.z & 0x0F0F0F0Fu) | ((hi.z & 0x0F0F0F0Fu) << 4);
        w[3] = (lo.w & 0x0F0F0F0Fu) | ((hi.w & 0x0F0F0F0Fu) << 4);
        put_bytes(y + 16 * j, w);
    } else if (j < 12) {
        // qh bytes 16 (j - 8) ..: the two high bits of elements li, li + 32, li + 64, li + 96 of a half block
        const int a = 8 * ((j - 8) >> 1) + (j & 1);
        uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const uint4 g = Q[a + 2 * s];
            w[0] |= ((g.x >> 4) & 0x03030303u) << (2 * s);
            w[1] |= ((g.y >> 4) & 0x03030303u) << (2 * s);
            w[2] |= ((g.z >> 4) & 0x03030303u) << (2 * s);
            w[3] |= ((g.w >> 4) & 0x03030303u) << (2 * s);
        }
        put_bytes(y + 128 + 16 * (j - 8), w);
    } else if (j == 12) {
        put16(y + 208, dh);
    }
    store_blocks<DT, PER>(img, nblocks, pl);
}

// Two-bit quants of a 256-element block, four elements 32 apart in one byte (Q2K, Q3K): chunk c < 4 of 16 bytes.
__device__ __forceinline__ void put_two_bits(const uint4 *Q, int c, uint8_t *p) {
    const int a = 8 * (c >> 1) + (c & 1);
    uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const uint4 g = Q[a + 2 * s];
        w[0] |= (g.x & 0x03030303u) << (2 * s);
        w[1] |= (g.y & 0x03030303u) << (2 * s);
        w[2] |= (g.z & 0x03030303u) << (2 * s);
        w[3] |= (g.w & 0x03030303u) << (2 * s);
    }
    put_bytes(p, w);
}

// Q2K (k_quants.rs:770-839): sixteen groups of sixteen, make_qkx1_quants with three levels, 4-bit scales and minima
__global__ void __launch_bounds__(kLanes) quantize_q2k(const float *__restrict__ src, int64_t nblocks, cq_planes pl) {
    constexpr int DT = CQ_DTYPE_Q2K, TS = Ggml<DT>::kSize, PER = kLanes / 16;
    const float Q4SCALE = 15.0f;
    __shared__ __align__(16) float lds[kLanes * 20];
    __shared__ __align__(16) uint4 quants[kLanes];
    const int t = threadIdx.x, blk = t >> 4, j = t & 15;
    float x[16];
    load_groups<16>(src, nblocks * 16, lds, x);
    float scale, min;
    make_qkx1_quants<16>(x, 3, scale, min);
    float max_scale = max_of_8(scale), max_min = max_of_8(min);
    max_scale = fmaxf(max_scale, dpp_f<kRowMirror>(max_scale));
    max_min = fmaxf(max_min, dpp_f<kRowMirror>(max_min));
    uint16_t dh = cq_f2h(0.0f), dmh = cq_f2h(0.0f);
    uint8_t sc = 0;
    if (max_scale > 0.0f) {
        const float iscale = Q4SCALE / max_scale;
        sc = (uint8_t)cq_nearest_int(iscale * scale);
        dh = cq_f2h(max_scale / Q4SCALE);
    }
    if (max_min > 0.0f) {
        const float iscale = Q4SCALE / max_min;
        sc |= (uint8_t)((uint8_t)cq_nearest_int(iscale * min) << 4);
        dmh = cq_f2h(max_min / Q4SCALE);
    }
    const float d = cq_h2f(dh) * (float)(sc & 0xF);
    int l[16];
#pragma unroll
    for (int i = 0; i < 16; i++) l[i] = 0;
    if (d != 0.0f) {
        const float dm = cq_h2f(dmh) * (float)(sc >> 4);
#pragma unroll
        for (int i = 0; i < 16; i++) l[i] = round_unsigned((x[i] + dm) / d, 3.0f);
    }
    quants[t] = pack16(l);
    __syncthreads();
    uint8_t *img = (uint8_t *)lds, *y = img + blk * TS;
    y[j] = sc;
    if (j < 4) put_two_bits(quants + blk * 16, j, y + 16 + 16 * j);
    else if (j == 4) put16(y + 80, dh);
    else if (j == 5) put16(y + 82, dmh);
    store_blocks<DT, PER>(img, nblocks, pl);
}

// utils.rs:261-326 with nmax = 4, do_rmse = true, n = 16: only the returned scale is used
__device__ __forceinline__ float make_q3_quants_16(const float (&x)[16]) {
    const int n = 16, nmax = 4;
    int l[16];
    float max = 0.0f, amax = 0.0f;
#pragma unroll
    for (int i = 0; i < n; i++) {
        const float ax = fabsf(x[i]);
        if (ax > amax) { amax = ax; max = x[i]; }
    }
    if (amax == 0.0f) return 0.0f;
    const float iscale = -(float)nmax / max;
    float sumlx = 0.0f, suml2 = 0.0f;
#pragma unroll
    for (int i = 0; i < n; i++) {
        l[i] = round_signed(iscale * x[i], -nmax, nmax - 1);
        const float w = x[i] * x[i];
        sumlx += w * x[i] * (float)l[i];
        suml2 += w * (float)(l[i] * l[i]);
    }
    for (int t = 0; t < 5; t++) {
        bool changed = false;
#pragma unroll
        for (int i = 0; i < n; i++) {
            const float w = x[i] * x[i];
            float slx = sumlx - w * x[i] * (float)l[i];
            if (slx > 0.0f) {
                float sl2 = suml2 - w * (float)(l[i] * l[i]);
                const int new_l = round_signed(x[i] * sl2 / slx, -nmax, nmax - 1);
                if (new_l != l[i]) {
                    slx += w * x[i] * (float)new_l;
                    sl2 += w * (float)(new_l * new_l);
                    if (sl2 > 0.0f && slx * slx * suml2 > sumlx * sumlx * sl2) {
                        l[i] = new_l;
                        sumlx = slx;
                        suml2 = sl2;
                        changed = true;
                    }
                }
            }
        }
        if (!changed) break;
    }
    return sumlx / suml2;
}

__global__ void __launch_bounds__(kLanes) quantize_q3k(const float *__restrict__ src, int64_t nblocks, cq_planes pl) {
    constexpr int DT = CQ_DTYPE_Q3K, TS = Ggml<DT>::kSize, PER = kLanes / 16;
    __shared__ __align__(16) float lds[kLanes * 20];
    __shared__ __align__(16) float scales[kLanes];
    __shared__ __align__(16) uint4 quants[kLanes];
    __shared__ __align__(16) uint8_t codes[kLanes];
    const int t = threadIdx.x, blk = t >> 4, j = t & 15;
    float x[16], all[16];
    load_groups<16>(src, nblocks * 16, lds, x);
    share_scales(scales, make_q3_quants_16(x), all);
    float max_scale = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i++)
        if (fabsf(all[i]) > fabsf(max_scale)) max_scale = all[i];
    uint16_t dh = cq_f2h(0.0f);
    int s6 = 0;   // the six-bit scale code as stored
    if (max_scale != 0.0f) {
        const float iscale = -32.0f / max_scale;
        s6 = cq_clampi(cq_nearest_int(iscale * scales[t]), -32, 31) + 32;
        dh = cq_f2h(1.0f / iscale);
    }
    codes[t] = (uint8_t)s6;
    const float d = cq_h2f(dh) * (float)(s6 - 32);
    int l[16];
#pragma unroll
    for (int i = 0; i < 16; i++) l[i] = 0;
    if (d != 0.0f) {
#pragma unroll
        for (int i = 0; i < 16; i++) l[i] = round_signed(x[i] / d, -4, 3) + 4;
    }
    quants[t] = pack16(l);
    __syncthreads();
    uint8_t *img = (uint8_t *)lds, *y = img + blk * TS;
    const uint4 *Q = quants + blk * 16;
    // element e: two low bits into qs[32 * (e / 128) + e % 32] at 2 * ((e % 128) / 32), the third into hmask[e % 32] bit e / 32
    if (j < 4) {
        put_two_bits(Q, j, y + 32 + 16 * j);
    } else if (j < 6) {
        uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const uint4 g = Q[(j & 1) + 2 * s];
            w[0] |= ((g.x >> 2) & 0x01010101u) << s;
            w[1] |= ((g.y >> 2) & 0x01010101u) << s;
            w[2] |= ((g.z >> 2) & 0x01010101u) << s;
            w[3] |= ((g.w >> 2) & 0x01010101u) << s;
        }
        put_bytes(y + 16 * (j & 1), w);
    } else if (j == 6) {
        const uint4 c = *(const uint4 *)(codes + blk * 16);   // codes 0..3, 4..7, 8..11, 12..15
        uint32_t w[3];
        w[0] = (c.x & 0x0F0F0F0Fu) | ((c.z & 0x0F0F0F0Fu) << 4);
        w[1] = (c.y & 0x0F0F0F0Fu) | ((c.w & 0x0F0F0F0Fu) << 4);
        w[2] = ((c.x >> 4) & 0x03030303u) | (((c.y >> 4) & 0x03030303u) << 2) | (((c.z >> 4) & 0x03030303u) << 4) |
               (((c.w >> 4) & 0x03030303u) << 6);
        put_bytes(y + 96, w);
    } else if (j == 7) {
        put16(y + 108, dh);
    }
    store_blocks<DT, PER>(img, nblocks, pl);
}

template <typename K> hipError_t launch(K kernel, const cq_weight *w, int lanes_per_block, const float *src, hipStream_t s) {
    const int64_t nblocks = w->n * (w->k / cq_block_size(w->ggml_dtype)), groups = nblocks * lanes_per_block;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((groups + kLanes - 1) / kLanes)), dim3(kLanes), 0, s, src, nblocks,
                       cq_planes{w->p0, w->p1, w->p2, w->p3, w->p4, w->p5});
    return hipGetLastError();
}

}  // namespace

hipError_t cq_launch_quantize_weight(const cq_weight *w, const float *src, hipStream_t s) {
    if (w->n == 0 || w->k == 0) return hipSuccess;
    switch (w->ggml_dtype) {
    case CQ_DTYPE_Q4_0: return launch(quantize_blk32<CQ_DTYPE_Q4_0>, w, 1, src, s);
    case CQ_DTYPE_Q4_1: return launch(quantize_blk32<CQ_DTYPE_Q4_1>, w, 1, src, s);
    case CQ_DTYPE_Q5_0: return launch(quantize_blk32<CQ_DTYPE_Q5_0>, w, 1, src, s);
    case CQ_DTYPE_Q5_1: return launch(quantize_blk32<CQ_DTYPE_Q5_1>, w, 1, src, s);
    case CQ_DTYPE_Q8_0: return launch(quantize_blk32<CQ_DTYPE_Q8_0>, w, 1, src, s);
    case CQ_DTYPE_Q4K: return launch(quantize_q4k<16>, w, 8, src, s);
    case CQ_DTYPE_Q5K: return launch(quantize_q4k<32>, w, 8, src, s);
    case CQ_DTYPE_Q2K: return launch(quantize_q2k, w, 16, src, s);
    case CQ_DTYPE_Q3K: return launch(quantize_q3k, w, 16, src, s);
    case CQ_DTYPE_Q6K: return launch(quantize_q6k, w, 16, src, s);
    default: return hipErrorInvalidValue;
    }
}
