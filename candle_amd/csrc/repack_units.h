// One unit of work of the byte permutation between a GGML block and the device planes, either way: repack_unit<DT, INVERSE>(x, b, u, planes)
// moves unit u < Ggml<DT>::kUnits of block b, whose GGML bytes lie at x (an even address; 16-byte aligned for Q4K and Q5K), in global memory
// or in LDS.  The units of a block may run in any order; in the inverse direction they write disjoint bytes of the block.
#pragma once
#include "qhip_internal.h"

template <int DT> struct Ggml;   // bytes of a block; units
template <> struct Ggml<CQ_DTYPE_Q4_0> { static constexpr int kSize = 18, kUnits = 1; };
template <> struct Ggml<CQ_DTYPE_Q4_1> { static constexpr int kSize = 20, kUnits = 1; };
template <> struct Ggml<CQ_DTYPE_Q5_0> { static constexpr int kSize = 22, kUnits = 1; };
template <> struct Ggml<CQ_DTYPE_Q5_1> { static constexpr int kSize = 24, kUnits = 1; };
template <> struct Ggml<CQ_DTYPE_Q8_0> { static constexpr int kSize = 34, kUnits = 1; };
template <> struct Ggml<CQ_DTYPE_Q4K> { static constexpr int kSize = 144, kUnits = 9; };
template <> struct Ggml<CQ_DTYPE_Q5K> { static constexpr int kSize = 176, kUnits = 10; };
template <> struct Ggml<CQ_DTYPE_Q6K> { static constexpr int kSize = 210, kUnits = 8; };
template <> struct Ggml<CQ_DTYPE_Q3K> { static constexpr int kSize = 110, kUnits = 8; };
template <> struct Ggml<CQ_DTYPE_Q2K> { static constexpr int kSize = 84, kUnits = 8; };

struct cq_planes { uint8_t *p0, *p1, *p2, *p3, *p4, *p5; };

#if defined(__HIPCC__)
namespace {

typedef uint32_t u32_any __attribute__((aligned(2)));                          // GGML blocks lie at even addresses
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(2)));
__device__ __forceinline__ void load16(const uint8_t *p, uint32_t (&v)[4]) {
    const u32x4_any x = *(const u32x4_any *)p;
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
}
__device__ __forceinline__ void store16(uint8_t *p, const uint32_t (&v)[4]) {
    u32x4_any x = {v[0], v[1], v[2], v[3]};
    *(u32x4_any *)p = x;
}
// bits 4i .. 4i+3 of `bits` as bit 0 of the four bytes of a word, and back
__device__ __forceinline__ uint32_t spread4(uint32_t bits, int i) {
    const uint32_t n = (bits >> (4 * i)) & 15u;
    return (n & 1u) | ((n & 2u) << 7) | ((n & 4u) << 14) | ((n & 8u) << 21);
}
__device__ __forceinline__ uint32_t gather4(uint32_t w, int i) {
    return ((w & 1u) | ((w >> 7) & 2u) | ((w >> 14) & 4u) | ((w >> 21) & 8u)) << (4 * i);
}

// The 16 header bytes {f16 d; f16 dmin; u8 scales[12]} of a Q4K / Q5K block <-> the 20-byte device
// record: the twelve bytes of 6-bit fields (utils.rs:49-59 get_scale_min_k4) unpacked to one byte
// per field and grouped per 32 qs bytes, record g = {sc[2g], sc[2g+1], mn[2g], mn[2g+1]}; the
// inverse packs them back (every one of the 96 bits is a field bit, so the round trip is exact).
template <bool INVERSE> __device__ __forceinline__ void k4_header(uint4 *a, uint32_t *h) {
    if constexpr (!INVERSE) {
        const uint4 v = *a;
        h[0] = v.x;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            int s0, m0, s1, m1;
            cq_scale_min_k4(2 * g, v.y, v.z, v.w, s0, m0);
            cq_scale_min_k4(2 * g + 1, v.y, v.z, v.w, s1, m1);
            h[1 + g] = (uint32_t)s0 | ((uint32_t)s1 << 8) | ((uint32_t)m0 << 16) | ((uint32_t)m1 << 24);
        }
    } else {
        uint32_t sc[8], mn[8];
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const uint32_t r = h[1 + g];
            sc[2 * g] = r & 0xff; sc[2 * g + 1] = (r >> 8) & 0xff;
            mn[2 * g] = (r >> 16) & 0xff; mn[2 * g + 1] = r >> 24;
        }
        uint32_t w[3] = {0, 0, 0};   // scales[0..3], scales[4..7], scales[8..11]
#pragma unroll
        for (int j = 0; j < 4; j++) {
            w[0] |= ((sc[j] & 63) | ((sc[j + 4] >> 4) << 6)) << (8 * j);
            w[1] |= ((mn[j] & 63) | ((mn[j + 4] >> 4) << 6)) << (8 * j);
            w[2] |= ((sc[j + 4] & 15) | ((mn[j + 4] & 15) << 4)) << (8 * j);
        }
        *a = make_uint4(h[0], w[0], w[1], w[2]);
    }
}

// ---- Q4K: 144-byte blocks {f16 d; f16 dmin; u8 scales[12]; u8 qs[128]}: unit 0 the header, units 1..8 sixteen bytes of nibbles ----
// ---- Q5K: 176-byte blocks {f16 d; f16 dmin; u8 scales[12]; u8 qh[32]; u8 qs[128]}: the same, unit 9 the whole qh ----
// (k_quants.rs:119-127).  Header and nibbles as Q4K.  Bit j of qh[l] is the fifth bit of element
// l of sub-block j, i.e. of the low (j even) or high (j odd) nibble of qs byte 32*(j/2) + l.  The
// device plane holds, per 32 qs bytes g, two words L (sub-block 2g) and H (sub-block 2g+1) with
//   bit 8c + i  =  fifth bit belonging to byte c of qs word i  (l = 4i + c),
// so that (W >> i) & 0x01010101 lines the four bits up with the four nibbles of word i.
template <int DT, bool INVERSE> __device__ __forceinline__ void k4_unit(uint8_t *x, int64_t b, int u, const cq_planes &pl) {
    constexpr int QS = DT == CQ_DTYPE_Q5K ? 48 : 16;
    if (u == 0) {
        k4_header<INVERSE>((uint4 *)x, (uint32_t *)(pl.p1 + b * CQ_Q4K_HDR));
    } else if (u <= 8) {
        uint4 *a = (uint4 *)(x + QS) + (u - 1), *p = (uint4 *)(pl.p0 + b * 128) + (u - 1);
        if constexpr (!INVERSE) *p = *a; else *a = *p;
    } else {
        uint4 *src = (uint4 *)(x + 16);              // GGML qh[32]
        uint4 *dst = (uint4 *)(pl.p2 + b * 32);      // {L, H} x 4
        // bit 8c + i of L_g = bit 2g of byte c of word i, bit 8c + i of H_g = bit 2g + 1: a transpose in words, its own form both ways
        const uint4 x0 = INVERSE ? dst[0] : src[0], x1 = INVERSE ? dst[1] : src[1];
        const uint32_t in[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
        uint32_t out[8];
#pragma unroll
        for (int o = 0; o < 8; o++) {
            out[o] = 0;
#pragma unroll
            for (int i = 0; i < 8; i++) out[o] |= ((in[i] >> o) & 0x01010101u) << i;
        }
        (INVERSE ? src : dst)[0] = make_uint4(out[0], out[1], out[2], out[3]);
        (INVERSE ? src : dst)[1] = make_uint4(out[4], out[5], out[6], out[7]);
    }
}

// ---- Q6K: 210-byte blocks {u8 ql[128]; u8 qh[64]; i8 scales[16]; f16 d} -----
// qh is re-ordered so that the thread that owns ql bytes [16u, 16u+16) of a block
// finds the high bits of exactly those 32 elements in qh' bytes [8u, 8u+8):
//   u = 4h + 2t + i  ->  ql byte 64h + 32t + 16i + e  (e < 16)
//   low  nibble: element 128h + 32t + 16i + e        hi bits = qh[32h + 16i + e] >> 2t
//   high nibble: element 128h + 64 + 32t + 16i + e   hi bits = qh[32h + 16i + e] >> (2t + 4)
//   qh'[8u + 4x + c] (x < 2, c < 4) =   lo2(8x + c)       | hi2(8x + c) << 2
//                                      | lo2(8x + 4 + c) << 4 | hi2(8x + 4 + c) << 6
//   sc'[2u], sc'[2u + 1] = scales[js], scales[js + 4] with js = u + 4h: the scales of the lane's
//   low-nibble and high-nibble 16-element groups, one 2-byte load per lane.
// i.e. for the two ql words 2x and 2x+1 of the lane, (H >> {0,2,4,6}) & 0x03030303 lines the
// two high bits up with each byte of {word 2x low, word 2x high, word 2x+1 low, word 2x+1 high}.
template <bool INVERSE> __device__ __forceinline__ void q6k_unit(uint8_t *x, int64_t b, int u, const cq_planes &pl) {
    const int h = u >> 2, tt = (u >> 1) & 1, i0 = (u & 1) * 16, js = u + 4 * h;
    uint4 *pql = (uint4 *)(pl.p0 + b * 128 + 16 * u);
    uint2 *pqh = (uint2 *)(pl.p1 + b * 64 + 8 * u);
    uint16_t *psc = (uint16_t *)(pl.p2 + b * 16) + u, *d = (uint16_t *)pl.p3;
    uint32_t q[4];
    if constexpr (!INVERSE) {
        load16(x + 16 * u, q);
        *pql = make_uint4(q[0], q[1], q[2], q[3]);
        load16(x + 128 + 32 * h + i0, q);
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = ((q[i] >> (2 * tt)) & 0x03030303u) | (((q[i] >> (2 * tt + 4)) & 0x03030303u) << 2);
        *pqh = make_uint2(q[0] | (q[1] << 4), q[2] | (q[3] << 4));
        // the lane's two 16-element scale groups (low nibbles: js, high nibbles: js + 4) side by side
        *psc = (uint16_t)(x[192 + js] | (x[192 + js + 4] << 8));
        if (u == 0) d[b] = *(const uint16_t *)(x + 208);
    } else {
        const uint4 v = *pql;
        q[0] = v.x; q[1] = v.y; q[2] = v.z; q[3] = v.w;
        store16(x + 16 * u, q);
        const uint16_t sc = *psc;
        x[192 + js] = (uint8_t)sc;
        x[192 + js + 4] = (uint8_t)(sc >> 8);
        if (u == 0) *(uint16_t *)(x + 208) = d[b];
        // Each GGML qh byte 32h + j collects 2-bit fields from the two units t = 0, 1 that share (h, i); unit (h, t = 0, i)
        // rebuilds the 16 bytes 32h + 16i + e from both units' qh'.
        if (tt == 0) {
            const uint2 v0 = pqh[0], v1 = pqh[2];
            const uint32_t a[2] = {v0.x, v0.y}, c[2] = {v1.x, v1.y};
#pragma unroll
            for (int i = 0; i < 4; i++) {   // element words 8x and 8x + 4: fields at bits 0-3 and 4-7
                const uint32_t f0 = a[i >> 1] >> (4 * (i & 1)), f1 = c[i >> 1] >> (4 * (i & 1));
                q[i] = (f0 & 0x03030303u) | ((f1 & 0x03030303u) << 2) | (((f0 >> 2) & 0x03030303u) << 4) | (((f1 >> 2) & 0x03030303u) << 6);
            }
            store16(x + 128 + 32 * h + i0, q);
        }
    }
}

// ---- Q4_0: 18-byte blocks {f16 d; u8 qs[16]}; Q8_0: 34-byte blocks {f16 d; i8 qs[32]} ----
template <int DT, bool INVERSE> __device__ __forceinline__ void blk32_unit(uint8_t *x, int64_t b, const cq_planes &pl) {
    constexpr int N = DT == CQ_DTYPE_Q8_0 ? 2 : 1;
    uint4 *p = (uint4 *)pl.p0 + b * N;
    uint16_t *d = (uint16_t *)pl.p1 + b;
#pragma unroll
    for (int i = 0; i < N; i++) {
        uint32_t q[4];
        if constexpr (!INVERSE) {
            load16(x + 2 + 16 * i, q);
            p[i] = make_uint4(q[0], q[1], q[2], q[3]);
        } else {
            const uint4 v = p[i];
            q[0] = v.x; q[1] = v.y; q[2] = v.z; q[3] = v.w;
            store16(x + 2 + 16 * i, q);
        }
    }
    if constexpr (!INVERSE) *d = *(const uint16_t *)x; else *(uint16_t *)x = *d;
}

// ---- types held in another type's planes: straight between the GGML blocks and the planes, in words of four quants ----
// In Q8_0 planes, one unit per block:
//   Q5_0 {f16 d; u8 qh[4]; u8 qs[16]} (k_quants.rs:61-67) holds d and 32 five-bit quants q, value d * (q - 16): exactly a
//   Q8_0 block {f16 d; i8 qs[32]} with qs = q - 16, whose dequantization (k_quants.rs:568-584) and dot product with Q8_0
//   activations (:631-649) are the arithmetic of Q5_0's (:428-451, :371-391) operation for operation.
//   Q4_1 {f16 d; f16 m; u8 qs[16]} and Q5_1 {f16 d; f16 m; u8 qh[4]; u8 qs[16]} (k_quants.rs:51-57, :69-76), value
//   d * q + m: the quants (0..15, 0..31) and d as a Q8_0 block, m into its own plane.
template <int DT, bool INVERSE>
__device__ __forceinline__ void held_in_q8_0(uint8_t *x, int64_t b, const cq_planes &pl) {
    constexpr bool FIVE = DT != CQ_DTYPE_Q4_1, MIN = DT != CQ_DTYPE_Q5_0;
    constexpr int QH = MIN ? 4 : 2, QS = FIVE ? QH + 4 : QH;
    constexpr uint32_t OFF = DT == CQ_DTYPE_Q5_0 ? 16 : 0;
    uint4 *p = (uint4 *)(pl.p0 + b * 32);
    uint16_t *d = (uint16_t *)pl.p1, *mins = (uint16_t *)pl.p2;
    uint32_t lo[4], hi[4];
    if constexpr (!INVERSE) {
        uint32_t q[4];
        load16(x + QS, q);
        const uint32_t qh = FIVE ? *(const u32_any *)(x + QH) : 0u;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            lo[i] = q[i] & 0x0F0F0F0Fu;
            hi[i] = (q[i] >> 4) & 0x0F0F0F0Fu;
            if (FIVE) {
                lo[i] |= spread4(qh, i) << 4;
                hi[i] |= spread4(qh, 4 + i) << 4;
            }
            if (OFF) {   // byte - 16 for bytes 0..31: + 0xF0 in each byte without its carry
                lo[i] = (lo[i] ^ 0x10101010u) | (((~lo[i] >> 4) & 0x01010101u) * 0xE0u);
                hi[i] = (hi[i] ^ 0x10101010u) | (((~hi[i] >> 4) & 0x01010101u) * 0xE0u);
            }
        }
        p[0] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        p[1] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        d[b] = *(const uint16_t *)x;
        if (MIN) mins[b] = *(const uint16_t *)(x + 2);
    } else {
        const uint4 a = p[0], c = p[1];
        lo[0] = a.x; lo[1] = a.y; lo[2] = a.z; lo[3] = a.w;
        hi[0] = c.x; hi[1] = c.y; hi[2] = c.z; hi[3] = c.w;
        uint32_t q[4], qh = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (OFF) {   // the low five bits of q - 16 are those of q with the fifth flipped
                lo[i] ^= 0x10101010u;
                hi[i] ^= 0x10101010u;
            }
            q[i] = (lo[i] & 0x0F0F0F0Fu) | ((hi[i] & 0x0F0F0F0Fu) << 4);
            if (FIVE) qh |= gather4(lo[i] >> 4, i) | gather4(hi[i] >> 4, 4 + i);
        }
        store16(x + QS, q);
        if (FIVE) *(u32_any *)(x + QH) = qh;
        *(uint16_t *)x = d[b];
        if (MIN) *(uint16_t *)(x + 2) = mins[b];
    }
}

// In Q6K planes, eight units per block, unit u = 4h + 2t + i the unit u of the Q6K layout above (ql bytes 16u ..: the
// elements 128h + 32t + 16i + e in the low and those 64 further on in the high nibbles):
//   Q3K {u8 hmask[32]; u8 qs[64]; u8 scales[12]; f16 d} (k_quants.rs:107-114): sixteen groups of sixteen three-bit quants,
//   value (d * (sc_j - 32)) * (q - 4) with six-bit sc_j: exactly a Q6K block {ql, qh, i8 scales[16], f16 d} with
//   scales[j] = sc_j - 32 and six-bit quants q + 28 (so that q6 - 32 = q - 4), whose dequantization (k_quants.rs:1716-1746)
//   and dot product with Q8K activations (:1585-1641) are those of Q3K (:1094-1146, :890-1009): the same integers, the
//   same products in the same order.
//   Q2K {u8 scales[16]; u8 qs[64]; f16 d; f16 dmin} (k_quants.rs:96-103): value (d * sc_j) * q - dmin * m_j, sc_j and m_j
//   the nibbles of scales[j].  The first term is a Q6K block with scales sc_j and quants q + 32; m_j and dmin go to planes
//   of their own.
// Both hold the two low bits of four elements 32 apart in one byte of qs[32h + 16i ..], at 2 * (element / 32 % 4); Q3K's
// third bit is bit element / 32 of hmask[16i ..].
__device__ __forceinline__ int q3k_scale6(const uint8_t *sc, int j) {
    const int low = j < 8 ? (sc[j] & 0xF) : (sc[j - 8] >> 4);
    return low | (((sc[8 + j % 4] >> (2 * (j / 4))) & 3) << 4);
}
// the six-bit quants of unit u (16 in the low, 16 in the high nibbles) out of the planes
__device__ __forceinline__ void q6_unit(const uint8_t *ql, const uint8_t *qh, int64_t b, int u, uint32_t (&lo)[4], uint32_t (&hi)[4]) {
    const uint4 q = *(const uint4 *)(ql + b * 128 + 16 * u);
    const uint2 H = *(const uint2 *)(qh + b * 64 + 8 * u);
    const uint32_t qw[4] = {q.x, q.y, q.z, q.w}, hw[2] = {H.x, H.y};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t f = hw[i >> 1] >> (4 * (i & 1));
        lo[i] = (qw[i] & 0x0F0F0F0Fu) | ((f & 0x03030303u) << 4);
        hi[i] = ((qw[i] >> 4) & 0x0F0F0F0Fu) | (((f >> 2) & 0x03030303u) << 4);
    }
}
template <int DT, bool INVERSE>
__device__ __forceinline__ void held_in_q6k(uint8_t *x, int64_t b, int u, const cq_planes &pl) {
    constexpr bool Q3 = DT == CQ_DTYPE_Q3K;
    constexpr int QS = Q3 ? 32 : 16, D = Q3 ? 108 : 80;
    constexpr uint32_t OFF = Q3 ? 0x1C1C1C1Cu : 0x20202020u;   // 28 or 32 in each byte
    const int h = u >> 2, t = (u >> 1) & 1, i16 = u & 1;
    uint8_t *ql = pl.p0, *qh = pl.p1, *sc = pl.p2, *mins = pl.p4;
    uint16_t *d = (uint16_t *)pl.p3, *dmins = (uint16_t *)pl.p5;
    if constexpr (!INVERSE) {
        uint32_t q[4], m[4] = {0, 0, 0, 0}, out[4], lo[4], hi[4];
        load16(x + QS + 32 * h + 16 * i16, q);
        if (Q3) load16(x + 16 * i16, m);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            lo[i] = ((q[i] >> (2 * t)) & 0x03030303u) + OFF;
            hi[i] = ((q[i] >> (2 * t + 4)) & 0x03030303u) + OFF;
            if (Q3) {
                lo[i] += ((m[i] >> (4 * h + t)) & 0x01010101u) << 2;
                hi[i] += ((m[i] >> (4 * h + t + 2)) & 0x01010101u) << 2;
            }
            out[i] = (lo[i] & 0x0F0F0F0Fu) | ((hi[i] & 0x0F0F0F0Fu) << 4);
            lo[i] = (lo[i] >> 4) & 0x03030303u;
            hi[i] = (hi[i] >> 4) & 0x03030303u;
        }
        *(uint4 *)(ql + b * 128 + 16 * u) = make_uint4(out[0], out[1], out[2], out[3]);
        *(uint2 *)(qh + b * 64 + 8 * u) = make_uint2(lo[0] | (hi[0] << 2) | (lo[1] << 4) | (hi[1] << 6),
                                                    lo[2] | (hi[2] << 2) | (lo[3] << 4) | (hi[3] << 6));
        const int js = u + 4 * h;
        if (Q3) {
            sc[b * 16 + 2 * u] = (uint8_t)(int8_t)(q3k_scale6(x + 96, js) - 32);
            sc[b * 16 + 2 * u + 1] = (uint8_t)(int8_t)(q3k_scale6(x + 96, js + 4) - 32);
        } else {
            const uint8_t s0 = x[js], s1 = x[js + 4];
            sc[b * 16 + 2 * u] = s0 & 0xF;
            sc[b * 16 + 2 * u + 1] = s1 & 0xF;
            mins[b * 16 + js] = s0 >> 4;
            mins[b * 16 + js + 4] = s1 >> 4;
        }
        if (u == 0) {
            d[b] = *(const uint16_t *)(x + D);
            if (!Q3) dmins[b] = *(const uint16_t *)(x + D + 2);
        }
        return;
    }
    uint32_t lo[4], hi[4];
    if (t == 0) {
        // qs[32h + 16i ..]: the units t = 0 (quarters 0 and 2) and t = 1 (1 and 3)
        uint32_t q[4], lo1[4], hi1[4];
        q6_unit(ql, qh, b, u, lo, hi);
        q6_unit(ql, qh, b, u + 2, lo1, hi1);
#pragma unroll
        for (int i = 0; i < 4; i++)
            q[i] = ((lo[i] - OFF) & 0x03030303u) | (((lo1[i] - OFF) & 0x03030303u) << 2) | (((hi[i] - OFF) & 0x03030303u) << 4) |
                   (((hi1[i] - OFF) & 0x03030303u) << 6);
        store16(x + QS + 32 * h + 16 * i16, q);
    } else if (Q3 && h == 0) {
        uint32_t m[4] = {0, 0, 0, 0};
#pragma unroll
        for (int v = 0; v < 4; v++) {   // the units of both halves and quarters with this i: bits 4h + t and 4h + t + 2
            q6_unit(ql, qh, b, 2 * v + i16, lo, hi);
            const int bit = 4 * (v >> 1) + (v & 1);
#pragma unroll
            for (int i = 0; i < 4; i++)
                m[i] |= ((((lo[i] - OFF) >> 2) & 0x01010101u) << bit) | ((((hi[i] - OFF) >> 2) & 0x01010101u) << (bit + 2));
        }
        store16(x + 16 * i16, m);
    } else if (u == 6) {   // h = 1, t = 1, i = 0: the scales (sc' holds group js = u + 4h at 2u and js + 4 at 2u + 1)
        uint8_t s[16];
#pragma unroll
        for (int v = 0; v < 8; v++) {
            s[v + 4 * (v >> 2)] = sc[b * 16 + 2 * v];
            s[v + 4 * (v >> 2) + 4] = sc[b * 16 + 2 * v + 1];
        }
        if (Q3) {
            uint8_t o[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const int lv = (int)(int8_t)s[j] + 32;
                o[j & 7] |= (uint8_t)((lv & 0xF) << (j < 8 ? 0 : 4));
                o[8 + j % 4] |= (uint8_t)((lv >> 4) << (2 * (j / 4)));
            }
#pragma unroll
            for (int j = 0; j < 12; j++) x[96 + j] = o[j];
        } else {
#pragma unroll
            for (int j = 0; j < 16; j++) x[j] = (uint8_t)((s[j] & 0xF) | (mins[b * 16 + j] << 4));
        }
    } else if (u == 7) {
        *(uint16_t *)(x + D) = d[b];
        if (!Q3) *(uint16_t *)(x + D + 2) = dmins[b];
    }
}

template <int DT, bool INVERSE> __device__ __forceinline__ void repack_unit(uint8_t *x, int64_t b, int u, const cq_planes &pl) {
    if constexpr (DT == CQ_DTYPE_Q4_0 || DT == CQ_DTYPE_Q8_0) blk32_unit<DT, INVERSE>(x, b, pl);
    else if constexpr (DT == CQ_DTYPE_Q5_0 || DT == CQ_DTYPE_Q4_1 || DT == CQ_DTYPE_Q5_1) held_in_q8_0<DT, INVERSE>(x, b, pl);
    else if constexpr (DT == CQ_DTYPE_Q4K || DT == CQ_DTYPE_Q5K) k4_unit<DT, INVERSE>(x, b, u, pl);
    else if constexpr (DT == CQ_DTYPE_Q6K) q6k_unit<INVERSE>(x, b, u, pl);
    else held_in_q6k<DT, INVERSE>(x, b, u, pl);
}

}  // namespace
#endif
