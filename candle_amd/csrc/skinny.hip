// Skinny matmul on int8 MFMA for a few activation rows (up to 32 to a workgroup; cq_qmatmul sends it 2..16 rows,
// more where the weight has few rows): y[m, n] = x[m, k] . W[n, k]^T with K-quant
// weights and Q8K activations (Q8_0 weights with Q8_0 activations: second kernel below) (k_quants.rs:1842-1883 with vec_dot :1171-1250 for Q4K, :1585-1641
// for Q6K) - the small-batch decode and the per-expert shapes of a mixture-of-experts layer, where
// the weights are still read once and the job stays bound by HBM.  The arithmetic is that of the
// prefill GEMM (gemm.hip): sub-block scales folded into the int8 weight operands as two digits,
// exact block integers I = 8*hi + lo (Q4K) / 128*hi + lo (Q5K, Q6K), the Q4K / Q5K min term on the f16 MFMA.
//
// Work split: with so few activation rows there is no tile to reuse weights over, so the K
// dimension is split instead.  A workgroup owns 16 weight rows (one 16x16x64 MFMA operand); its
// eight waves take the 256-element K blocks round-robin (wave w: blocks w, w+8, ...).  Per block a
// wave copies its 16 x 144 (210) weight bytes and the block's activation slice from global memory
// straight into its own LDS buffer (buffer_load ... lds, whole 128-byte lines, XOR-swizzled as in
// gemm.hip), unpacks, and issues eight MFMAs per 16 activation rows.  The waves' partial 16 x 16
// results are summed through LDS in wave order (deterministic; no atomics).  Many small workgroups
// (n / 16) and one block in flight per wave keep enough bytes outstanding per CU.
#include "quantize_blocks.h"

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
// the same at four-byte alignment: scales of 32-element blocks in rows of no whole 256 elements
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned short us2 __attribute__((ext_vector_type(2)));
typedef short ss2 __attribute__((ext_vector_type(2)));
typedef const void __attribute__((address_space(1))) *gptr_t;
typedef void __attribute__((address_space(3))) *lptr_t;

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
// First weight row of 16-row tile `t`: the last tile of an n that is no multiple of 16 begins at row n - 16, on top of the
// tile before it (both store the same values there).
__device__ __forceinline__ int64_t tile_row(int64_t t, int64_t n) { return t * 16 + 16 <= n ? t * 16 : n - 16; }

constexpr int kMaxLds = 160 * 1024;   // LDS of a CU, which a single workgroup may take

// both 16-bit halves of `a` times `b` (a splat: the packed instruction takes one half of its operand twice)
__device__ __forceinline__ uint32_t pk_mul_u16(uint32_t a, unsigned short b) {
    const us2 r = __builtin_bit_cast(us2, a) * (us2){b, b};
    return __builtin_bit_cast(uint32_t, r);
}

// Buffer descriptor over `base` (wave-uniform): raw bytes, no stride, no bounds.  The copies below
// are buffer loads rather than global loads on purpose: with a global (FLAT-encoded) LDS copy in
// flight the compiler treats the LDS counter as out of order and turns every wait on an operand
// read into a wait for all of them, which serialises the software-pipelined LDS reads; a buffer
// load leaves the LDS counter alone and takes its per-lane offset without 64-bit vector adds.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t wave_rsrc(const void *base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, -1, 0x00020000);
}

__device__ __forceinline__ void dma16(const void *base, uint32_t off, uint8_t *lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(wave_rsrc(base), (lptr_t)lds, 16, (int)off, 0, 0, 0);
}
__device__ __forceinline__ void dma4(const void *base, uint32_t off, uint8_t *lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(wave_rsrc(base), (lptr_t)lds, 4, (int)off, 0, 0, 0);
}

// Per-wave LDS buffer for RT groups of eight activation rows:
//   wgt : [2 row groups][8 rows][8 chunks of 16 B] of the 128-byte qs / ql plane, chunk c of row r at c ^ (r%8);
//         Q6K also [16 rows][4 chunks] of the 64-byte qh plane (chunk c at c ^ ((r/2)%4)),
//         Q5K also [16 rows][32 B] of the fifth-bit plane
//   act : [RT row groups][2 K-halves][8 rows][8 chunks], same swizzle
//   d8  : [8*RT] f32         bsh : [8*RT][16] f16: the rows' bsums (Q4K / Q5K)
constexpr bool is_k4(int dt) { return dt == CQ_DTYPE_Q4K || dt == CQ_DTYPE_Q5K; }   // types with a min term

template <int DT, int RT> struct Buf {
    static constexpr int kWgt = DT == CQ_DTYPE_Q4K ? 2048 : DT == CQ_DTYPE_Q5K ? 2560 : 3072;
    static constexpr int oAct = kWgt, kAct = RT * 2048;
    static constexpr int oD8 = oAct + kAct, kD8 = RT * 32;
    static constexpr int oMin = oD8 + kD8, kMin = is_k4(DT) ? RT * 256 : 0;
    static constexpr int kRaw = oMin + kMin;
    // the buffer also carries the wave's partial results at the end: 1 KiB per 16 activation rows
    static constexpr int kBytes = kRaw < 2048 ? 2048 : kRaw;
};

__device__ __forceinline__ uint32_t swz_col(uint32_t r, uint32_t c) {
    return (r >> 3) * 1024u + (r & 7) * 128u + ((c ^ (r & 7)) << 4);
}

template <int DT> struct WHead;
template <> struct WHead<CQ_DTYPE_Q4K> { uint32_t dd; uint4 rec; };   // d | dmin << 16; records {sc, sc, mn, mn} per 32 qs bytes
template <> struct WHead<CQ_DTYPE_Q5K> : WHead<CQ_DTYPE_Q4K> {};       // the same header plane
template <> struct WHead<CQ_DTYPE_Q6K> { uint4 sc; uint32_t d; };     // re-packed scales (two per unit); d
__device__ __forceinline__ void load_head(const cq_weight &w, int64_t blk, WHead<CQ_DTYPE_Q4K> &r) {
    // two loads (16 + 4 bytes; the 20-byte records are 4-byte aligned, which is all a global load needs)
    typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
    const uint8_t *h = w.p1 + blk * CQ_Q4K_HDR;
    const u32x4_a4 v = *(const u32x4_a4 *)h;
    r.dd = v.x;
    r.rec = make_uint4(v.y, v.z, v.w, *(const uint32_t *)(h + 16));
}
__device__ __forceinline__ void load_head(const cq_weight &w, int64_t blk, WHead<CQ_DTYPE_Q6K> &r) {
    r.sc = *(const uint4 *)(w.p2 + blk * 16);
    r.d = ((const uint16_t *)w.p3)[blk];
}

// An empty statement that may change the fields (in the registers their loads came to, four at once).
__device__ __forceinline__ void hold_head(WHead<CQ_DTYPE_Q4K> &r) {
    v4i v = {(int)r.dd, (int)r.rec.x, (int)r.rec.y, (int)r.rec.z};
    asm volatile("" : "+v"(v), "+v"(r.rec.w));
    r.dd = (uint32_t)v.x;
    r.rec.x = (uint32_t)v.y;
    r.rec.y = (uint32_t)v.z;
    r.rec.z = (uint32_t)v.w;
}
__device__ __forceinline__ void hold_head(WHead<CQ_DTYPE_Q6K> &r) {
    v4i v = __builtin_bit_cast(v4i, r.sc);
    asm volatile("" : "+v"(v), "+v"(r.d));
    r.sc = __builtin_bit_cast(uint4, v);
}

// Weight operands of one block for lane (row r = l%16, k quarter kq = l/16): the two digit operands
// of the four 64-wide K-slices, the block scale and the Q4K min-term operand.
__device__ __forceinline__ void block_unpack(const uint8_t *wl, int lane, const WHead<CQ_DTYPE_Q4K> &wb, v4i (&bl)[4],
                                             v4i (&bh)[4], float &dw, v8h &wmin) {
    const uint32_t r = lane & 15, kq = lane >> 4;
    dw = cq_h2f((uint16_t)(wb.dd & 0xffff));
    const uint32_t rec[4] = {wb.rec.x, wb.rec.y, wb.rec.z, wb.rec.w};
    // K-slice g = elements 64g..64g+63 = qs bytes 32g..32g+31, low nibbles for the first 32 elements
    // (quarters 0,1: sub-block 2g), high nibbles for the last 32 (quarters 2,3: sub-block 2g+1)
    const uint32_t hi = kq >> 1, nsh = hi * 4;
#pragma unroll
    for (int gi = 0; gi < 4; gi++) {
        const uint4 q = *(const uint4 *)(wl + swz_col(r, 2 * gi + (kq & 1)));
        const uint32_t sj = (rec[gi] >> (8 * hi)) & 0xff;   // scale of sub-block 2g + hi
        const unsigned short sl = (unsigned short)(sj & 7), sh = (unsigned short)(sj >> 3);
        const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t v = (qw[i] >> nsh) & 0x0F0F0F0Fu;
            bl[gi][i] = (int)pk_mul_u16(v, sl);   // low digit of the scale
            bh[gi][i] = (int)pk_mul_u16(v, sh);
        }
    }
    // min term operand: 32 K-slots = activation pieces [1,1,2,2] x weight pieces [1,2,1,2] of the
    // eight sub-block values -dmin*min_j
    wmin = __builtin_bit_cast(v8h, cq_min_term_groups(wb.dd, rec, (kq & 1) != 0, (kq >> 1) != 0));   // K-slots 8kq..: groups 8(kq%2).., piece kq/2
}

// Q5K: the quants are the Q4K nibbles plus a fifth bit (words {L, H} per 32 qs bytes, bit 8c + i for
// byte c of qs word i); scale times quant has up to 11 bits and is split as Q6K's products are.
__device__ __forceinline__ void block_unpack(const uint8_t *wl, int lane, const WHead<CQ_DTYPE_Q5K> &wb, v4i (&bl)[4],
                                             v4i (&bh)[4], float &dw, v8h &wmin) {
    const uint32_t r = lane & 15, kq = lane >> 4;
    dw = cq_h2f((uint16_t)(wb.dd & 0xffff));
    const uint32_t rec[4] = {wb.rec.x, wb.rec.y, wb.rec.z, wb.rec.w};
    const uint32_t hi = kq >> 1, nsh = hi * 4, w0 = 4 * (kq & 1);   // first qs word of the lane's 16 bytes
    const uint4 f0 = *(const uint4 *)(wl + 2048 + r * 32u), f1 = *(const uint4 *)(wl + 2048 + r * 32u + 16u);
    const uint32_t fifth[4] = {hi ? f0.y : f0.x, hi ? f0.w : f0.z, hi ? f1.y : f1.x, hi ? f1.w : f1.z};
#pragma unroll
    for (int gi = 0; gi < 4; gi++) {
        const uint4 q = *(const uint4 *)(wl + swz_col(r, 2 * gi + (kq & 1)));
        const unsigned short sc16 = (unsigned short)((rec[gi] >> (8 * hi)) & 0xff);   // scale of sub-block 2g + hi
        const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t q5 = ((qw[i] >> nsh) & 0x0F0F0F0Fu) | (((fifth[gi] >> (w0 + i)) & 0x01010101u) << 4);
            int lo, hi;
            cq_scaled_digits(q5, sc16, (unsigned short)128, lo, hi);   // digits of sc * q5
            bl[gi][i] = lo;
            bh[gi][i] = hi;
        }
    }
    wmin = __builtin_bit_cast(v8h, cq_min_term_groups(wb.dd, rec, (kq & 1) != 0, (kq >> 1) != 0));   // K-slots 8kq..: groups 8(kq%2).., piece kq/2
}

__device__ __forceinline__ void block_unpack(const uint8_t *wl, int lane, const WHead<CQ_DTYPE_Q6K> &wb, v4i (&bl)[4],
                                             v4i (&bh)[4], float &dw, v8h &wmin) {
    const uint32_t r = lane & 15, kq = lane >> 4;
    dw = cq_h2f((uint16_t)wb.d);
#pragma unroll
    for (int hf = 0; hf < 2; hf++) {
        // K-slices 2hf (low nibbles) and 2hf+1 (high nibbles) of unit u = 4hf + kq: 16 bytes of ql,
        // 8 bytes of re-packed high bits, scale bytes 2u and 2u+1
        const uint4 ql = *(const uint4 *)(wl + swz_col(r, 4 * hf + kq));
        const uint2 qh = *(const uint2 *)(wl + 2048 + r * 64u + (((2 * hf + (kq >> 1)) ^ ((r >> 1) & 3)) << 4) + (kq & 1) * 8u);
        const uint32_t s_even = hf ? wb.sc.z : wb.sc.x, s_odd = hf ? wb.sc.w : wb.sc.y;
        const uint32_t sw = s_even ^ ((s_even ^ s_odd) & (0u - (kq >> 1)));   // word 2hf + kq/2, branch-free
        const uint32_t qw[4] = {ql.x, ql.y, ql.z, ql.w};
        const uint32_t hw[2] = {qh.x, qh.y};
#pragma unroll
        for (int nib = 0; nib < 2; nib++) {
            const int s = 2 * hf + nib;
            const int sc = (int)(int8_t)((sw >> (16 * (kq & 1) + 8 * nib)) & 0xff);
            const unsigned short sc16 = (unsigned short)sc, c16 = (unsigned short)(128 - 32 * sc);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t H = hw[i >> 1];
                const int sh = (i & 1) * 4 + 2 * nib;   // where the two high bits sit in H's bytes; wanted at bit 4
                const uint32_t hb = sh < 4 ? H << (4 - sh) : H >> (sh - 4);
                const uint32_t q6 = ((qw[i] >> (4 * nib)) & 0x0F0F0F0Fu) | (hb & 0x30303030u);
                int lo, hi;
                cq_scaled_digits(q6, sc16, c16, lo, hi);   // digits of sc * (q6 - 32)
                bl[s][i] = lo;
                bh[s][i] = hi;
            }
        }
    }
    wmin = v8h{};
}

// ---- the offset terms (min_term.hip), added to the result tiles of the waves ----
// A launch of its own for them is 4 of the 10 us of a call of a few rows (whole calls, launch on the vector units -> here: Q4_1 4096 x 4096 with
// 8 rows 23.2 -> 8.6, 11008 x 4096 30.2 -> 17.9, 1792 x 1792 with 5 rows 14.4 -> 7.1, Q2K 4096 x 4096 with 8 rows 13.9 -> 9.0).  out[t] += a step of 32 blocks' m * s products for the types held in
// Q8_0 planes, -= a block's dmin term for Q2K: the same products, exact in f32, on the same operands as there.  `first` and `stride` deal the
// steps to the waves.  Instances of their own (OFF), so that the kernels of the plain Q8_0 and
// Q6K weights keep their registers.
template <int NT>
__device__ __forceinline__ void add_min32(const cq_weight &w, const cq_act_view &a, int64_t n_tile, int64_t m0, int64_t m, int64_t first,
                                          int64_t stride, int lane, v4f (&out)[NT]) {
    const uint32_t r = lane & 15, kq = lane >> 4;
    const int64_t nb = w.k >> 5;
#pragma nounroll
    for (int64_t b0 = first * 32; b0 < nb; b0 += stride * 32) {
        const int64_t b = b0 + 8 * kq;   // (rows have an even number of blocks: pairs of 16-bit values start on a word)
        uint32_t mw[4];
        const uint32_t *mp = (const uint32_t *)w.p2 + (((n_tile + r) * nb + b) >> 1);
#pragma unroll
        for (int i = 0; i < 4; i++) mw[i] = b + 2 * i < nb ? mp[i] : 0u;
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int64_t row = m0 + t * 16 + r < m ? m0 + t * 16 + r : m - 1;
            const uint32_t *sp = (const uint32_t *)a.bsum32 + ((row * nb + b) >> 1);
            const float *dp = a.d + row * nb + b;
            v8h sv;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const bool in = b + 2 * i < nb;
                const uint32_t s = in ? sp[i] : 0u;
                const float d0 = in ? dp[2 * i] : 0.0f, d1 = in ? dp[2 * i + 1] : 0.0f;
                sv[2 * i] = (_Float16)((float)(_Float16)(float)(int16_t)s * d0);
                sv[2 * i + 1] = (_Float16)((float)(_Float16)(float)(int16_t)(s >> 16) * d1);
            }
            out[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(sv, __builtin_bit_cast(v8h, mw), out[t], 0, 0, 0);
        }
    }
}
template <int NT>
__device__ __forceinline__ void add_min16(const cq_weight &w, const cq_act_view &a, int64_t n_tile, int64_t m0, int64_t first, int64_t stride,
                                          int lane, v4f (&out)[NT]) {
    const uint32_t r = lane & 15, kq = lane >> 4;
    const int64_t kb = w.k >> 8;
#pragma nounroll
    for (int64_t b = first; b < kb; b += stride) {
        const int64_t blk = (n_tile + r) * kb + b;
        const uint32_t mq = *(const uint32_t *)(w.p4 + blk * 16 + 4 * kq);   // minima 4kq .. of the lane's weight row
        const float dm = cq_h2f(((const uint16_t *)w.p5)[blk]);
        v4h mv;
#pragma unroll
        for (int i = 0; i < 4; i++) mv[i] = (_Float16)(float)((mq >> (8 * i)) & 0xff);
#pragma unroll
        for (int t = 0; t < NT; t++) {   // (rows past the last one are the workspace's padding)
            const v4h sv = *(const v4h *)(a.bsh + (b * a.m_stride + m0 + t * 16 + r) * 16 + 4 * kq);
            const v4f d8 = *(const v4f *)(a.dT + b * a.m_stride + m0 + t * 16 + 4 * kq);
            const v4f sum = __builtin_amdgcn_mfma_f32_16x16x16f16(sv, mv, (v4f){0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; i++) out[t][i] -= (d8[i] * dm) * sum[i];
        }
    }
}

// The wave's rows of K block b, four at a time (lane l: row 4p + l/16, elements 64i + 4(l%16) ..; rows past m repeat the last one).
template <int RT>
__device__ __forceinline__ void load_direct(const float *__restrict__ x, int64_t m, int64_t k, int64_t b, int lane, float4 (&xf)[2 * RT][4]) {
#pragma unroll
    for (int p = 0; p < 2 * RT; p++) {
        if (4 * p >= m) continue;
        const int64_t row = 4 * p + (lane >> 4) < m ? 4 * p + (lane >> 4) : m - 1;
        const float *src = x + row * k + b * 256 + 4 * (lane & 15);
#pragma unroll
        for (int i = 0; i < 4; i++) xf[p][i] = *(const float4 *)(src + 64 * i);
    }
}
// ... quantized into the wave's buffer, in the image the copies of quantized rows make; `keep`: into the workspace as well.
template <int DT, int RT>
__device__ __forceinline__ void quantize_direct(const float4 (&xf)[2 * RT][4], const cq_act_view &a, int64_t m0, int64_t m, int64_t k, int64_t b, int lane,
                                                bool keep, uint8_t *buf) {
    typedef Buf<DT, RT> B;
    const int l = lane & 15;
    const uint32_t sj = 4 * (l & 3) + (l >> 2);   // the sum cq_q8k_of_sixteen leaves with this lane
#pragma unroll
    for (int p = 0; p < 2 * RT; p++) {
        if (4 * p >= m) continue;
        uint32_t packed[4];
        float d;
        int bsum;
        cq_q8k_of_sixteen(xf[p], l, packed, d, bsum);
        const uint32_t row = 4 * p + (lane >> 4);
        if (row >= m) continue;
        uint8_t *at = buf + B::oAct + (row >> 3) * 2048u + (row & 7) * 128u + (l & 3) * 4;
#pragma unroll
        for (int i = 0; i < 4; i++) *(uint32_t *)(at + (i >> 1) * 1024 + ((((i & 1) * 4 + (l >> 2)) ^ (row & 7)) << 4)) = packed[i];
        if (l == 0) *(float *)(buf + B::oD8 + row * 4) = d;
        if (is_k4(DT)) *(_Float16 *)(buf + B::oMin + row * 32 + sj * 2) = (_Float16)(float)bsum;
        if (keep) {
            const int64_t to = m0 + row, blk = to * (k >> 8) + b, tb = b * a.m_stride + to;
#pragma unroll
            for (int i = 0; i < 4; i++) *(uint32_t *)(a.qs + to * k + b * 256 + 64 * i + 4 * l) = packed[i];
            if (l == 0) {
                a.d[blk] = d;
                a.dT[tb] = d;
            }
            a.bsums[blk * 16 + sj] = (int16_t)bsum;
            ((_Float16 *)a.bsh)[tb * 16 + sj] = (_Float16)(float)bsum;
        }
    }
}

// RT = groups of eight activation rows held (rows m0 .. m0 + 8*RT - 1; the workspace pads rows, so
// whole groups can be copied); results are stored for rows < m.  Requires n >= 16.
// DUMP (verification): the block integers, and the min term as the f16 MFMA delivers it from a zero accumulator,
// are stored through `dump` instead of the result through `y`.
// DIRECT: the rows come as f32 from `x` and every wave quantizes the blocks it contracts (see skinny_direct_kernel).
template <int DT, int RT, bool DUMP, bool DIRECT = false, int NW = kWaves, bool OFF = false>
__device__ __forceinline__ void skinny_body(const cq_weight &w, const cq_act_view &a, int64_t tile, int64_t m0, int64_t m,
                                            float *__restrict__ y, cq_mfma_dump dump, const float *__restrict__ x = nullptr) {
    typedef Buf<DT, RT> B;
    constexpr bool MINS = is_k4(DT);
    constexpr int NT = (RT + 1) / 2;   // 16-row tiles
    constexpr int SHIFT = DT == CQ_DTYPE_Q4K ? 3 : 8;
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r = lane & 15, kq = lane >> 4;
    const int64_t k = w.k, kb = w.k >> 8;
    const int64_t n_tile = tile_row(tile, w.n);
    uint8_t *buf = smem + wave * B::kBytes;

    // copy offsets: 8 rows x 128 B per instruction, chunks swizzled by the row
    const uint32_t r8 = lane >> 3, c8 = lane & 7;
    const uint32_t act_off = r8 * (uint32_t)k + ((c8 ^ r8) << 4);
    const uint32_t wq_off = r8 * (uint32_t)kb * 128u + ((c8 ^ r8) << 4);
    const uint32_t r16 = lane >> 2, c4 = lane & 3;
    const uint32_t wh_off = r16 * (uint32_t)kb * 64u + ((c4 ^ ((r16 >> 1) & 3)) << 4);
    const uint32_t w5_off = (lane >> 1) * (uint32_t)kb * 32u + (lane & 1) * 16u;   // Q5K: 16 rows x 32 B, lanes 0..31
    // activation operand reads: row of tile t clamped to the rows held
    uint32_t a_col[NT][2];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const uint32_t row = t * 16 + r < 8u * RT ? t * 16 + r : 8u * RT - 1;
#pragma unroll
        for (uint32_t e = 0; e < 2; e++)
            a_col[t][e] = B::oAct + (row >> 3) * 2048u + (row & 7) * 128u + (((4 * e + kq) ^ (row & 7)) << 4);
    }

    v4f out[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) out[t] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};

    for (int64_t b = wave; b < kb; b += NW) {
        // ---- copies of block b: weights of the 16 rows, activation rows, their scales
        float4 xf[DIRECT ? 2 * RT : 1][4];
        if constexpr (DIRECT) {
            load_direct<RT>(x + m0 * k, m - m0, k, b, lane, xf);   // (first: what the quantizer waits for; requests are answered in order)
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int rg = 0; rg < 2; rg++) dma16(w.p0 + ((n_tile + rg * 8) * kb + b) * 128, wq_off, buf + rg * 1024);
        if (DT == CQ_DTYPE_Q6K) dma16(w.p1 + (n_tile * kb + b) * 64, wh_off, buf + 2048);
        if (DT == CQ_DTYPE_Q5K && lane < 32) dma16(w.p2 + (n_tile * kb + b) * 32, w5_off, buf + 2048);
        if constexpr (!DIRECT) {
#pragma unroll
        for (int i = 0; i < 2 * RT; i++) {
            const int rg = i >> 1, kh = i & 1;
            if (RT > 1 || (int64_t)r8 < m - m0)   // (few rows: the others' copies are most of the activations')
                dma16(a.qs + (m0 + rg * 8) * k + b * 256 + kh * 128, act_off, buf + B::oAct + i * 1024);
        }
        if (lane < 8 * RT) dma4(a.dT + b * a.m_stride + m0, lane * 4u, buf + B::oD8);
        if (MINS && lane < 16 * RT) dma16(a.bsh + (b * a.m_stride + m0) * 16, lane * 16u, buf + B::oMin);
        }
        WHead<DT> head;
        load_head(w, (n_tile + r) * kb + b, head);
        if constexpr (DIRECT) {
            __builtin_amdgcn_sched_barrier(0);
            quantize_direct<DT, RT>(xf, a, m0, m - m0, k, b, lane, tile == 0, buf);
        }
        __builtin_amdgcn_s_waitcnt(0);   // everything above has landed

        // ---- arithmetic of block b
        v4i bl[4], bh[4];
        float dw;
        v8h wmin;
        block_unpack(buf, lane, head, bl, bh, dw, wmin);
        if constexpr (DUMP && is_k4(DT)) {
            if (dump.int_min) {   // verification: the minima themselves as the operand: the MFMA delivers the integer Mn_b
                const uint32_t rec[4] = {head.rec.x, head.rec.y, head.rec.z, head.rec.w};
                wmin = __builtin_bit_cast(v8h, cq_min_term_groups_int(rec, (kq & 1) != 0, (kq >> 1) != 0));
            }
        }
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const v4f d8 = *(const v4f *)(buf + B::oD8 + (t * 16 + 4 * kq < 8u * RT ? t * 16 + 4 * kq : 0) * 4);
            // min term: sum_j bsums_j * (-dmin * min_{j/2}), the sums exact in f16 whatever the activations' magnitude
            // (their scale d8 multiplies afterwards, with the main term)
            v4f mn = {0.0f, 0.0f, 0.0f, 0.0f};
            if (MINS) {
                const uint32_t row = t * 16 + r < 8u * RT ? t * 16 + r : 8u * RT - 1;
                const v8h ma = *(const v8h *)(buf + B::oMin + row * 32 + (kq & 1) * 16);
                mn = __builtin_amdgcn_mfma_f32_16x16x32_f16(ma, wmin, mn, 0, 0, 0);
                if (DUMP && dump.mn) {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int64_t orow = m0 + t * 16 + kq * 4 + i;
                        if (orow < m) dump.mn[(orow * w.n + n_tile + r) * kb + b] = mn[i];
                    }
                }
            }
            v4i acc_lo = {0, 0, 0, 0}, acc_hi = {0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const v4i av = *(const v4i *)(buf + a_col[t][s & 1] + (s >> 1) * 1024);
                acc_lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bl[s], acc_lo, 0, 0, 0);
                acc_hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bh[s], acc_hi, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int I = (acc_hi[i] << SHIFT) + acc_lo[i];
                if (DUMP) {
                    const int64_t orow = m0 + t * 16 + kq * 4 + i;
                    if (orow < m) dump.i[(orow * w.n + n_tile + r) * kb + b] = I;
                } else {
                    const float v = MINS ? __builtin_fmaf((float)I, dw, mn[i]) : (float)I * dw;
                    out[t][i] = __builtin_fmaf(v, d8[i], out[t][i]);
                }
            }
        }
    }
    if (DUMP) return;
    if constexpr (OFF) add_min16<NT>(w, a, n_tile, m0, wave, NW, lane, out);

    // ---- sum the waves' partial tiles in wave order
#pragma unroll
    for (int t = 0; t < NT; t++) *(v4f *)(buf + t * 1024 + lane * 16) = out[t];
    __syncthreads();
    if (wave < NT) {
        v4f s = *(const v4f *)(smem + wave * 1024 + lane * 16);
#pragma unroll
        for (int o = 1; o < NW; o++) {
            const v4f p = *(const v4f *)(smem + o * B::kBytes + wave * 1024 + lane * 16);
            s += p;
        }
        const int64_t col = n_tile + r;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int64_t row = m0 + wave * 16 + kq * 4 + i;
            if (row < m) y[row * w.n + col] = s[i];
        }
    }
}

template <int DT, int RT, bool DUMP, int NW = kWaves, bool OFF = false>
__global__ void __launch_bounds__(NW * 64) skinny_kernel(cq_weight w, cq_act_view a, int64_t m0, int64_t m, float *__restrict__ y,
                                                          cq_mfma_dump dump) {
    skinny_body<DT, RT, DUMP, false, NW, OFF>(w, a, blockIdx.x, m0 + blockIdx.y * (8 * RT), m, y, dump);   // (a group of rows for each y)
}

// ------------------------------------------------------------ resident-activation variant ----
// The kernel above re-reads the activations once per 16 weight rows: with 16 activation rows that is more
// bytes (from L2) than the weights themselves (16 K against 9 K per workgroup for Q4K), and the launch is bound
// by it.  When the quantized activations of the call fit the LDS beside the weight buffers (4096 columns x 16
// rows: 75 KiB) a launch of at most one workgroup per CU copies them once, each wave the K blocks it owns (sixteen
// waves: one block each for 4096 columns, a single memory round trip).  The launcher takes it where every
// workgroup has one 16-row weight tile (n <= 16 x the number of CUs); walking several tiles measured no faster than
// the kernel above, also with the next tile's weights copied ahead into a second buffer.  The loop over tiles cost registers that sixteen
// waves do not have, and spills with 17 rows and more (whole calls from a graph, weights from HBM, us, with it -> without, 4096 x 4096: 24 rows
// Q4K 10.7 -> 9.4, Q5K 14.2 -> 9.9, Q2K 12.6 -> 11.2; 8 rows Q2K 10.0 -> 9.7; Q4K, Q5K and Q6K with 8 and 16 rows level).
//   per K block b  : act [RT][2 K-halves][8 rows][8 chunks] | d8 [8*RT] f32 | bsh [8*RT][16] f16 (k4 types)
//   per K block    : weights (kWgt bytes); a wave's first buffer also carries its partial results (1 KiB per 16 activation rows)
template <int DT, int RT> struct Res {
    static constexpr int kWgt = Buf<DT, RT>::kWgt;
    static constexpr int kActBlk = RT * 2048 + RT * 32 + (is_k4(DT) ? RT * 256 : 0);
    static constexpr int oD8 = RT * 2048, oMin = oD8 + RT * 32;
    static size_t bytes(int64_t kb) { return (size_t)kb * (kActBlk + kWgt); }
};

// Copies with one descriptor per plane, built once, and the position inside the plane as a 32-bit scalar offset
// (the planes of a tensor this kernel takes are far below 4 GiB): two scalar instructions per copy instead of
// rebuilding a descriptor from a 64-bit address for each.
struct ResPlanes {
    __amdgpu_buffer_rsrc_t wq, wh, w5, aq, ad, am;
};
__device__ __forceinline__ void dma16s(__amdgpu_buffer_rsrc_t rs, uint32_t voff, uint32_t soff, uint8_t *lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lptr_t)lds, 16, (int)voff, (int)soff, 0, 0);
}
__device__ __forceinline__ void dma4s(__amdgpu_buffer_rsrc_t rs, uint32_t voff, uint32_t soff, uint8_t *lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lptr_t)lds, 4, (int)voff, (int)soff, 0, 0);
}

// Issues the copies of the weights of the tile starting at row n_tile for K block b into `wl`.
template <int DT>
__device__ __forceinline__ void res_issue_weights(uint8_t *__restrict__ wl, const ResPlanes &pl, uint32_t n_tile, uint32_t b,
                                                  uint32_t kb, uint32_t wq_off, uint32_t wh_off, uint32_t w5_off, int lane) {
    const uint32_t blk = n_tile * kb + b;
    dma16s(pl.wq, wq_off, blk * 128u, wl);
    dma16s(pl.wq, wq_off, blk * 128u + kb * 1024u, wl + 1024);
    if (DT == CQ_DTYPE_Q6K) dma16s(pl.wh, wh_off, blk * 64u, wl + 2048);
    if (DT == CQ_DTYPE_Q5K && lane < 32) dma16s(pl.w5, w5_off, blk * 32u, wl + 2048);
}

// Weight operands of one K block of one tile, unpacked into registers.
struct ResOps {
    v4i bl[4], bh[4];
    float dw;
    v8h wmin;
};
template <int DT, bool DUMP>
__device__ __forceinline__ void res_unpack(const uint8_t *__restrict__ wl, int lane, const WHead<DT> &head, const cq_mfma_dump &dump,
                                           ResOps &o) {
    block_unpack(wl, lane, head, o.bl, o.bh, o.dw, o.wmin);
    if constexpr (DUMP && is_k4(DT)) {
        if (dump.int_min) {   // verification: the minima themselves as the operand: the MFMA delivers the integer Mn_b
            const uint32_t kq = lane >> 4;
            const uint32_t rec[4] = {head.rec.x, head.rec.y, head.rec.z, head.rec.w};
            o.wmin = __builtin_bit_cast(v8h, cq_min_term_groups_int(rec, (kq & 1) != 0, (kq >> 1) != 0));
        }
    }
}

// The unpacked operands `o` contracted with the resident activation slice `act` of the same K block.
// DUMP: the integers go to dump.i / dump.mn at `at` + row * `rs` (rows < m) instead of into `out`.
template <int DT, int RT, int NT, bool DUMP>
__device__ __forceinline__ void res_mac(const uint8_t *__restrict__ act, int lane, const ResOps &o, const uint32_t (&a_col)[NT][2],
                                        v4f (&out)[NT], const cq_mfma_dump &dump, int64_t at, int64_t rs, int64_t m) {
    typedef Res<DT, RT> R;
    constexpr bool MINS = is_k4(DT);
    constexpr int SHIFT = DT == CQ_DTYPE_Q4K ? 3 : 8;
    const uint32_t r = lane & 15, kq = lane >> 4;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const v4f d8 = *(const v4f *)(act + R::oD8 + (t * 16 + 4 * kq < 8u * RT ? t * 16 + 4 * kq : 0) * 4);
        v4f mn = {0.0f, 0.0f, 0.0f, 0.0f};   // min term without the activation scale (see skinny_kernel)
        if (MINS) {
            const uint32_t row = t * 16 + r < 8u * RT ? t * 16 + r : 8u * RT - 1;
            const v8h ma = *(const v8h *)(act + R::oMin + row * 32 + (kq & 1) * 16);
            mn = __builtin_amdgcn_mfma_f32_16x16x32_f16(ma, o.wmin, mn, 0, 0, 0);
            if (DUMP && dump.mn) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int64_t orow = t * 16 + kq * 4 + i;
                    if (orow < m) dump.mn[at + orow * rs] = mn[i];
                }
            }
        }
        v4i acc_lo = {0, 0, 0, 0}, acc_hi = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const v4i av = *(const v4i *)(act + a_col[t][s & 1] + (s >> 1) * 1024);
            acc_lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, o.bl[s], acc_lo, 0, 0, 0);
            acc_hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, o.bh[s], acc_hi, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int I = (acc_hi[i] << SHIFT) + acc_lo[i];
            if (DUMP) {
                const int64_t orow = t * 16 + kq * 4 + i;
                if (orow < m) dump.i[at + orow * rs] = I;
            } else {
                const float v = MINS ? __builtin_fmaf((float)I, o.dw, mn[i]) : (float)I * o.dw;
                out[t][i] = __builtin_fmaf(v, d8[i], out[t][i]);
            }
        }
    }
}

// One K block of one tile: unpack the weights in `wl`, contract with the resident activation slice `act`.
template <int DT, int RT, int NT, bool DUMP>
__device__ __forceinline__ void res_block(const uint8_t *__restrict__ wl, const uint8_t *__restrict__ act, int lane,
                                          const WHead<DT> &head, const uint32_t (&a_col)[NT][2], v4f (&out)[NT],
                                          const cq_mfma_dump &dump, int64_t at, int64_t rs, int64_t m) {
    ResOps o;
    res_unpack<DT, DUMP>(wl, lane, head, dump, o);
    res_mac<DT, RT, NT, DUMP>(act, lane, o, a_col, out, dump, at, rs, m);
}

// m <= 8 * RT activation rows (the workspace pads rows, so whole groups are copied); n >= 16, one 16-row tile per workgroup; at most
// kMaxBpw K blocks per wave.
constexpr int kMaxBpw = 4;
template <int DT, int RT, int kWaves, bool DUMP, bool OFF = false>
__global__ void __launch_bounds__(kWaves * 64) skinny_resident_kernel(cq_weight w, cq_act_view a, int64_t m,
                                                                      float *__restrict__ y, cq_mfma_dump dump) {
    typedef Res<DT, RT> R;
    constexpr bool MINS = is_k4(DT);
    constexpr int NT = (RT + 1) / 2;   // 16-row tiles of activation rows
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r = lane & 15, kq = lane >> 4;
    const int64_t k = w.k, kb = w.k >> 8;
    const int64_t n_tile = tile_row(blockIdx.x, w.n);
    uint8_t *wgt_base = smem + kb * R::kActBlk;

    const uint32_t r8 = lane >> 3, c8 = lane & 7;
    const uint32_t act_off = r8 * (uint32_t)k + ((c8 ^ r8) << 4);
    const uint32_t wq_off = r8 * (uint32_t)kb * 128u + ((c8 ^ r8) << 4);
    const uint32_t r16 = lane >> 2, c4 = lane & 3;
    const uint32_t wh_off = r16 * (uint32_t)kb * 64u + ((c4 ^ ((r16 >> 1) & 3)) << 4);
    const uint32_t w5_off = (lane >> 1) * (uint32_t)kb * 32u + (lane & 1) * 16u;
    uint32_t a_col[NT][2];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const uint32_t row = t * 16 + r < 8u * RT ? t * 16 + r : 8u * RT - 1;
#pragma unroll
        for (uint32_t e = 0; e < 2; e++)
            a_col[t][e] = (row >> 3) * 2048u + (row & 7) * 128u + (((4 * e + kq) ^ (row & 7)) << 4);
    }
    ResPlanes pl;
    pl.wq = wave_rsrc(w.p0);
    pl.wh = wave_rsrc(w.p1);
    pl.w5 = wave_rsrc(w.p2);
    pl.aq = wave_rsrc(a.qs);
    pl.ad = wave_rsrc(a.dT);
    pl.am = wave_rsrc(a.bsh);
    const uint32_t kb32 = (uint32_t)kb, k32 = (uint32_t)k, mstr = (uint32_t)a.m_stride;
    // ---- the wave's K blocks: the small fields of the weights (registers; requested first, they are what the unpacking
    // starts with), activation slices, weights
    WHead<DT> head[kMaxBpw];
#pragma unroll
    for (int j = 0; j < kMaxBpw; j++) {
        const int64_t b = wave + (int64_t)j * kWaves;
        if (b < kb) load_head(w, (n_tile + r) * kb + b, head[j]);
    }
#pragma unroll
    for (int j = 0; j < kMaxBpw; j++) {
        const uint32_t b = (uint32_t)wave + (uint32_t)j * kWaves;
        if (b < kb32) {
            uint8_t *act = smem + b * R::kActBlk;
#pragma unroll
            for (int i = 0; i < 2 * RT; i++) {
                const uint32_t rg = i >> 1, kh = i & 1;
                dma16s(pl.aq, act_off, rg * 8u * k32 + b * 256u + kh * 128u, act + i * 1024);
            }
            if (lane < 8 * RT) dma4s(pl.ad, lane * 4u, b * mstr * 4u, act + R::oD8);
            if (MINS && lane < 16 * RT) dma16s(pl.am, lane * 16u, b * mstr * 32u, act + R::oMin);
            res_issue_weights<DT>(wgt_base + b * R::kWgt, pl, (uint32_t)n_tile, b, kb32, wq_off, wh_off, w5_off, lane);
        }
    }
    v4f out[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) out[t] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    // One pass of a loop whose count the compiler does not know: what does not depend on the data (addresses in the images, the lane's masks) is
    // then formed in front of it, while the copies are on their way, and not behind the wait in each block that uses it.  The block fields
    // change in the loop as far as the compiler can see, so that nothing made of them moves in front and waits for them there.  (Without the
    // loop, weights from HBM: Q6K 4096 x 4096 with 8 rows 9.0 -> 9.3 us, with 24 10.1 -> 10.2, Q4K 4096 x 2048 6.7 -> 6.9.)
    int passes = 1;
    asm volatile("" : "+s"(passes));
    for (int pass = 0; pass < passes; pass++) {
        __builtin_amdgcn_s_waitcnt(0);   // everything above has landed
#pragma unroll
        for (int j = 0; j < kMaxBpw; j++) {
            const int64_t b = wave + (int64_t)j * kWaves;
            if (b < kb) {
                hold_head(head[j]);
                res_block<DT, RT, NT, DUMP>(wgt_base + b * R::kWgt, smem + b * R::kActBlk, lane, head[j], a_col, out, dump, (n_tile + r) * kb + b, w.n * kb, m);
            }
        }
    }
    if (DUMP) return;
    if constexpr (OFF) {
        if (wave < kb) add_min16<NT>(w, a, n_tile, 0, wave, kb < kWaves ? kb : kWaves, lane, out);
    }
    // ---- sum the waves' partial tiles in wave order (through each wave's first weight buffer)
    if (wave < kb) {   // (a wave without a K block has no buffer and nothing to add)
        uint8_t *part = wgt_base + (int64_t)wave * R::kWgt;
#pragma unroll
        for (int t = 0; t < NT; t++) *(v4f *)(part + t * 1024 + lane * 16) = out[t];
    }
    __syncthreads();
    if (wave < NT) {
        v4f s = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
        const int64_t nw = kb < kWaves ? kb : kWaves;   // waves that own a block
        for (int64_t o = 0; o < nw; o++) {
            const v4f p = *(const v4f *)(wgt_base + o * R::kWgt + wave * 1024 + lane * 16);
            s += p;
        }
        const int64_t col = n_tile + r;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int64_t row = wave * 16 + kq * 4 + i;
            if (row < m) y[row * w.n + col] = s[i];
        }
    }
}

// ------------------------------------------- resident activations, several tiles per workgroup ----
// More weight rows than 16 x the number of CUs: every workgroup walks several 16-row tiles.  With one K block per
// wave (k <= 256 x waves) a wave keeps its partial result of each tile in registers and the workgroup meets once per
// round of up to four tiles, not once per tile: between two tiles of a round there is no barrier and no wait for
// the slowest wave, so the copies of the tile after the next one (issued into the buffer the current tile has just
// been unpacked from) really are in flight under the arithmetic.  Everything a tile needs comes through LDS copies,
// the 20-byte block headers included: a load into registers would be tracked by the compiler, which on joining the
// paths "copies issued" and "no tile left to copy" waits as the stricter of the two demands, i.e. for everything.
// The waits are written out by hand instead (s_waitcnt vmcnt(copies of one tile) while a next tile is in flight).
// The partial tiles of a round are summed in wave order as in the kernels above.  Q4K and Q5K (one header layout).
//   LDS: activation slices as skinny_resident_kernel | per wave two slots {weights kWgt | headers 16 x 16 B, 16 x 4 B},
//        which take the wave's partial results (1 KiB per tile) at the end of a round
constexpr int kTilesPerRound = 4;
template <int DT, int RT> struct ResMulti {
    static constexpr int kWgt = Res<DT, RT>::kWgt;
    static constexpr int oHdr = kWgt, kSlot = kWgt + 320;
    static constexpr int kCopies = (DT == CQ_DTYPE_Q4K ? 2 : 3) + 2;   // copy instructions per tile (multi_issue)
    static size_t bytes(int64_t kb) { return (size_t)kb * Res<DT, RT>::kActBlk + (size_t)kb * 2 * kSlot; }
};

constexpr int kMultiMax = 3;
struct MultiArgs {
    cq_weight w[kMultiMax];
    float *y[kMultiMax];
    uint32_t first[kMultiMax];   // first tile of the launch that is the weight's
};
// Where a tile of the launch lies: its weight's planes and first row.  One weight, or two or three with the same rows (skinny_shared_kernel).
struct TileAt {
    const uint8_t *p0, *p1, *p2;
    float *y;
    int64_t n;
    uint32_t row;
};
struct OneWeight {
    const cq_weight &w;
    float *y;
    __device__ int64_t k() const { return w.k; }
    __device__ int64_t tiles() const { return (w.n + 15) / 16; }
    __device__ TileAt at(int64_t t) const { return {w.p0, w.p1, w.p2, y, w.n, (uint32_t)tile_row(t, w.n)}; }
};
struct SomeWeights {
    const MultiArgs &ma;
    uint32_t total;
    __device__ int64_t k() const { return ma.w[0].k; }
    __device__ int64_t tiles() const { return total; }
    __device__ TileAt at(int64_t t) const {
        const bool b = t >= ma.first[1], c = t >= ma.first[2];
        const auto pick = [&](auto x, auto y, auto z) { return c ? z : b ? y : x; };
        const int64_t n = pick(ma.w[0].n, ma.w[1].n, ma.w[2].n);
        return {pick(ma.w[0].p0, ma.w[1].p0, ma.w[2].p0), pick(ma.w[0].p1, ma.w[1].p1, ma.w[2].p1), pick(ma.w[0].p2, ma.w[1].p2, ma.w[2].p2),
                pick(ma.y[0], ma.y[1], ma.y[2]), n, (uint32_t)tile_row(t - pick(ma.first[0], ma.first[1], ma.first[2]), n)};
    }
};

// The copies of one tile's K block b into `slot`: weights as res_issue_weights, then the 16 rows' headers
// (bytes 0..15 of row r at oHdr + 16 r, bytes 16..19 at oHdr + 256 + 4 r; lanes 0..15).
template <int DT, int RT>
__device__ __forceinline__ void multi_issue(uint8_t *__restrict__ slot, const TileAt &at, uint32_t b, uint32_t kb, uint32_t wq_off, uint32_t w5_off, uint32_t hd_off, int lane) {
    typedef ResMulti<DT, RT> M;
    ResPlanes pl;
    pl.wq = wave_rsrc(at.p0);
    pl.w5 = wave_rsrc(at.p2);
    const __amdgpu_buffer_rsrc_t hdr = wave_rsrc(at.p1);
    res_issue_weights<DT>(slot, pl, at.row, b, kb, wq_off, 0, w5_off, lane);
    const uint32_t blk = at.row * kb + b;
    if (lane < 16) {
        dma16s(hdr, hd_off, blk * (uint32_t)CQ_Q4K_HDR, slot + M::oHdr);
        // (the instruction's immediate offset moves both addresses: bytes 16.. of the header, and 16 bytes on in LDS)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(hdr, (lptr_t)(slot + M::oHdr + 256 - 16), 4, (int)hd_off, (int)(blk * (uint32_t)CQ_Q4K_HDR), 16, 0);
    }
}

// One tile of one wave: operands out of `slot`, then (the slot is free) the copies of the tile two ahead, then the MFMAs.
template <int DT, int RT, bool DUMP>
__device__ __forceinline__ void multi_step(uint8_t *__restrict__ slot, const uint8_t *__restrict__ act, int lane, bool ahead,
                                           const TileAt &next, uint32_t b, uint32_t kb32,
                                           uint32_t wq_off, uint32_t w5_off, uint32_t hd_off, const uint32_t (&a_col)[1][2],
                                           v4f (&out)[1], const cq_mfma_dump &dump, int64_t at, int64_t rs, int64_t m) {
    typedef ResMulti<DT, RT> M;
    const uint32_t r = lane & 15;
    WHead<DT> head;
    const uint4 h4 = *(const uint4 *)(slot + M::oHdr + r * 16u);
    head.dd = h4.x;
    head.rec = make_uint4(h4.y, h4.z, h4.w, *(const uint32_t *)(slot + M::oHdr + 256 + r * 4u));
    ResOps o;
    res_unpack<DT, DUMP>(slot, lane, head, dump, o);
    if (ahead) {
        __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the reads above are done with the slot
        multi_issue<DT, RT>(slot, next, b, kb32, wq_off, w5_off, hd_off, lane);
    }
    res_mac<DT, RT, 1, DUMP>(act, lane, o, a_col, out, dump, at, rs, m);
}

// m <= 8 * RT <= 16 activation rows; n >= 16; k / 256 <= kWaves.
template <int DT, int RT, int kWaves, bool DUMP, typename Set>
__device__ __forceinline__ void resident_rounds(const Set &set, const cq_act_view &a, int64_t m, const cq_mfma_dump &dump) {
    typedef Res<DT, RT> R;
    typedef ResMulti<DT, RT> M;
    static_assert(DT == CQ_DTYPE_Q4K || DT == CQ_DTYPE_Q5K, "block headers of 20 bytes");
    static_assert(RT <= 2, "one 16-row tile of activation rows");
    static_assert(2 * M::kSlot >= kTilesPerRound * 1024, "a round's partial tiles fit the wave's two slots");
    constexpr bool MINS = is_k4(DT);
    constexpr int kAhead = 0x0F70 | M::kCopies;   // s_waitcnt vmcnt(copies of one tile)
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r = lane & 15, kq = lane >> 4;
    const int64_t k = set.k(), kb = k >> 8;
    const int64_t tiles = set.tiles(), G = gridDim.x;
    uint8_t *wgt_base = smem + kb * R::kActBlk;
    const bool has = wave < kb;   // this wave owns K block `wave`
    const uint32_t b = (uint32_t)wave;

    const uint32_t r8 = lane >> 3, c8 = lane & 7;
    const uint32_t act_off = r8 * (uint32_t)k + ((c8 ^ r8) << 4);
    const uint32_t wq_off = r8 * (uint32_t)kb * 128u + ((c8 ^ r8) << 4);
    const uint32_t w5_off = (lane >> 1) * (uint32_t)kb * 32u + (lane & 1) * 16u;
    const uint32_t hd_off = (uint32_t)lane * (uint32_t)kb * (uint32_t)CQ_Q4K_HDR;   // lanes 0..15: the header of row `lane`
    uint32_t a_col[1][2];
    {
        const uint32_t row = r < 8u * RT ? r : 8u * RT - 1;
#pragma unroll
        for (uint32_t e = 0; e < 2; e++) a_col[0][e] = (row >> 3) * 2048u + (row & 7) * 128u + (((4 * e + kq) ^ (row & 7)) << 4);
    }
    ResPlanes pl;
    pl.aq = wave_rsrc(a.qs);
    pl.ad = wave_rsrc(a.dT);
    pl.am = wave_rsrc(a.bsh);
    const uint32_t kb32 = (uint32_t)kb, k32 = (uint32_t)k, mstr = (uint32_t)a.m_stride;
    uint8_t *act = smem + b * R::kActBlk;
    uint8_t *ring = wgt_base + (size_t)b * 2 * M::kSlot;

    // ---- the wave's activation slice, once
    if (has) {
#pragma unroll
        for (int i = 0; i < 2 * RT; i++) {
            const uint32_t rg = i >> 1, kh = i & 1;
            dma16s(pl.aq, act_off, rg * 8u * k32 + b * 256u + kh * 128u, act + i * 1024);
        }
        if (lane < 8 * RT) dma4s(pl.ad, lane * 4u, b * mstr * 4u, act + R::oD8);
        if (MINS && lane < 16 * RT) dma16s(pl.am, lane * 16u, b * mstr * 32u, act + R::oMin);
    }
    for (int64_t t0 = blockIdx.x; t0 < tiles; t0 += kTilesPerRound * G) {
        // tiles of this round: t0, t0 + G, ... (cnt of them)
        int cnt = (int)((tiles - t0 + G - 1) / G);
        cnt = cnt < kTilesPerRound ? cnt : kTilesPerRound;
        if (has) {
            v4f o0 = {0.0f, 0.0f, 0.0f, 0.0f}, o1 = o0, o2 = o0, o3 = o0;
            multi_issue<DT, RT>(ring, set.at(t0), b, kb32, wq_off, w5_off, hd_off, lane);
            if (cnt > 1) multi_issue<DT, RT>(ring + M::kSlot, set.at(t0 + G), b, kb32, wq_off, w5_off, hd_off, lane);
#pragma nounroll
            for (int i = 0; i < cnt; i++) {
                // everything but the copies of the next tile has landed
                if (i + 1 < cnt) __builtin_amdgcn_s_waitcnt(kAhead);
                else __builtin_amdgcn_s_waitcnt(0x0F70);
                const int64_t tile = t0 + i * G;
                v4f acc[1] = {{0.0f, 0.0f, 0.0f, 0.0f}};
                const TileAt here = set.at(tile);   // (for the dump)
                multi_step<DT, RT, DUMP>(ring + (i & 1) * M::kSlot, act, lane, i + 2 < cnt, set.at(i + 2 < cnt ? tile + 2 * G : tile), b, kb32, wq_off,
                                         w5_off, hd_off, a_col, acc, dump, ((int64_t)here.row + r) * kb + b, here.n * kb, m);
                // (i is wave-uniform: real branches, four moves, instead of sixteen selects - the empty statements keep them)
                if (i == 0) { o0 = acc[0]; asm volatile(""); }
                else if (i == 1) { o1 = acc[0]; asm volatile(""); }
                else if (i == 2) { o2 = acc[0]; asm volatile(""); }
                else { o3 = acc[0]; asm volatile(""); }
            }
            // ---- the round's partial tiles into the wave's slots (every copy into them has landed and been unpacked)
            *(v4f *)(ring + lane * 16) = o0;
            *(v4f *)(ring + 1024 + lane * 16) = o1;
            *(v4f *)(ring + 2048 + lane * 16) = o2;
            *(v4f *)(ring + 3072 + lane * 16) = o3;
        }
        __syncthreads();
        if (wave < cnt && !DUMP) {   // wave i sums tile i of the round, in wave order
            v4f s = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
            const int64_t nw = kb < kWaves ? kb : kWaves;   // waves that own a block
            for (int64_t o = 0; o < nw; o++) {
                const v4f p = *(const v4f *)(wgt_base + (size_t)o * 2 * M::kSlot + wave * 1024 + lane * 16);
                s += p;
            }
            const TileAt at = set.at(t0 + wave * G);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int64_t row = kq * 4 + i;
                if (row < m) at.y[row * at.n + at.row + r] = s[i];
            }
        }
        if (t0 + kTilesPerRound * G < tiles) __syncthreads();   // the sums have been read: the slots take the next round's copies
    }
}
template <int DT, int RT, int kWaves, bool DUMP>
__global__ void __launch_bounds__(kWaves * 64) skinny_resident_multi_kernel(cq_weight w, cq_act_view a, int64_t m, float *__restrict__ y,
                                                                            cq_mfma_dump dump) {
    resident_rounds<DT, RT, kWaves, DUMP>(OneWeight{w, y}, a, m, dump);
}
__global__ void __launch_bounds__(16 * 64) skinny_shared_rounds_kernel(MultiArgs ma, uint32_t tiles, cq_act_view a, int64_t m) {
    resident_rounds<CQ_DTYPE_Q4K, 2, 16, false>(SomeWeights{ma, tiles}, a, m, cq_mfma_dump{nullptr, nullptr, 0});
}

// ---------------------------------------------------- Q8_0 / Q4_0 weights x Q8_0 activations ----
// The same work split for 32-element blocks (k_quants.rs:618-649, :224-254: sumf += sumi * d_w *
// d_x per block).  Q8_0 weights are int8 already and Q4_0 weights become q - 8 with two instructions a word, so the
// operands go from LDS (almost) straight into the 16x16x32 MFMA, one per block, and each block's
// 16 x 16 integers are scaled by the two block scales on the way into the f32 result.  A wave
// takes 256 elements (eight blocks) per step.
// The activation scales come block-major (cq_act_view::dT), one LDS copy per group of eight rows and one 16-byte read per
// block for a lane's four result rows.  (Row-major they took a 16-byte request per result row and half step from every
// lane - 8 KiB of requests a step against 4 KiB of Q8_0 weights, twice that for Q4_0 with its block sums.)
//   wgt : Q8_0 [2 row groups][2 K-halves][8 rows][8 chunks of 16 B], Q4_0 [2 row groups][8 rows][8 chunks
//         = blocks]; chunk c of row r at c ^ (r%8)
//   act : [RT row groups][2 K-halves][8 rows][8 chunks], same swizzle
//   d8  : [RT row groups][8 blocks][8 rows] f32
template <int DT, int RT> struct BufQ8 {
    static constexpr int oAct = DT == CQ_DTYPE_Q8_0 ? 4096 : 2048, oD8 = oAct + RT * 2048, kRaw = oD8 + RT * 256;
    static constexpr int kBytes = kRaw;   // >= 1 KiB of partial results per 16 rows
};

// Activation scales of K step g for the rows m0 .. m0 + 8*RT - 1 into `lds` (row groups of 256 bytes).
template <int RT> __device__ __forceinline__ void issue_scales(const cq_act_view &a, int64_t m0, int64_t g, uint8_t *lds, int lane) {
    const uint32_t off = ((uint32_t)(lane >> 3) * (uint32_t)a.m_stride + (lane & 7)) * 4u;
#pragma unroll
    for (int rg = 0; rg < RT; rg++) dma4(a.dT + g * 8 * a.m_stride + m0 + rg * 8, off, lds + rg * 256);
}
// Where a lane finds the scales of result rows 4kq .. 4kq + 3 of tile t (+ 32 bytes per block); rows past the held groups
// repeat the last group (they are not stored).
template <int RT> __device__ __forceinline__ uint32_t scale_col(int t, uint32_t kq) {
    const uint32_t rg = 2 * t + (kq >> 1) < RT ? 2 * t + (kq >> 1) : RT - 1;
    return rg * 256u + (kq & 1) * 16u;
}
// Eight weight bytes of block b for the 16x16x32 MFMA out of a tile's LDS image.
template <bool Q4> __device__ __forceinline__ long weight_bytes(const uint8_t *wl, int b, uint32_t r, uint32_t w4_col, uint32_t w4_shift, const uint32_t (&w_col)[4]) {
    if (!Q4) return *(const long *)(wl + w_col[b & 3] + (b >> 2) * 1024);
    const uint2 raw = *(const uint2 *)(wl + w4_col + (((uint32_t)b ^ (r & 7)) << 4));
    // every byte minus 8, no carries between bytes
    const uint32_t lo = (((raw.x >> w4_shift) & 0x0F0F0F0Fu) + 0x78787878u) ^ 0x80808080u;
    const uint32_t hi = (((raw.y >> w4_shift) & 0x0F0F0F0Fu) + 0x78787878u) ^ 0x80808080u;
    return (long)(((uint64_t)hi << 32) | lo);
}

// The eight blocks of a 256-element step, or the `left` that a row ends with (left is wave-uniform; the copies of such a step
// also bring in what follows the row in memory, which nothing reads).
template <typename F> __device__ __forceinline__ void each_block(int64_t left, F block) {
    if (left >= 8) {
#pragma unroll
        for (int b = 0; b < 8; b++) block(b);
    } else {
#pragma unroll
        for (int b = 0; b < 7; b++)
            if (b < left) block(b);
    }
}

// The wave's rows of K step g for the bodies that quantize themselves (lane l: elements 4l .. of the step; zeros past the row's end).
template <int RT>
__device__ __forceinline__ void load_direct_q8(const float *__restrict__ x, int64_t m, int64_t k, int64_t g, int lane, float4 (&xf)[8 * RT]) {
    const int64_t e0 = g * 256 + 4 * lane;
#pragma unroll
    for (int row = 0; row < 8 * RT; row++) xf[row] = row < m && e0 < k ? *(const float4 *)(x + row * k + e0) : make_float4(0.f, 0.f, 0.f, 0.f);
}
template <int DT, int RT>
__device__ __forceinline__ void quantize_direct_q8(const float4 (&xf)[8 * RT], const cq_act_view &a, int64_t m0, int64_t m, int64_t k, int64_t g, int lane,
                                                   bool keep, uint8_t *buf) {
    typedef BufQ8<DT, RT> B;
    const int64_t e0 = g * 256 + 4 * lane;
#pragma unroll
    for (int row = 0; row < 8 * RT; row++) {
        if (row >= m) continue;
        uint32_t packed;
        float d;
        int sum;
        cq_q8_0_of_eight(xf[row], packed, d, sum);
        const float dr = cq_h2f(cq_f2h(d));
        *(uint32_t *)(buf + B::oAct + (row >> 3) * 2048 + (lane >> 5) * 1024 + (row & 7) * 128 + ((((lane >> 2) & 7) ^ (row & 7)) << 4) + (lane & 3) * 4) = packed;
        if ((lane & 7) == 0) *(float *)(buf + B::oD8 + (row >> 3) * 256 + (lane >> 3) * 32 + (row & 7) * 4) = dr;
        if (keep && e0 < k) {
            const int64_t to = m0 + row;
            *(uint32_t *)(a.qs + to * k + e0) = packed;
            if ((lane & 7) == 0) {
                const int64_t blk = to * (k >> 5) + (e0 >> 5);
                a.d[blk] = dr;
                a.bsum32[blk] = (int16_t)sum;
                a.dT[(e0 >> 5) * a.m_stride + to] = dr;
            }
        }
    }
}

template <int DT, int RT, bool DUMP, bool DIRECT = false, int NW = kWaves, bool OFF = false>
__device__ __forceinline__ void skinny_blk32_body(const cq_weight &w, const cq_act_view &a, int64_t tile, int64_t m0, int64_t m,
                                                  float *__restrict__ y, cq_mfma_dump dump, const float *__restrict__ x = nullptr) {
    typedef BufQ8<DT, RT> B;
    constexpr bool Q4 = DT == CQ_DTYPE_Q4_0;
    constexpr int NT = (RT + 1) / 2;   // 16-row tiles
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r = lane & 15, kq = lane >> 4;
    const int64_t k = w.k, kg = (w.k + 255) >> 8, kb = w.k >> 5;
    const int64_t n_tile = tile_row(tile, w.n);
    uint8_t *buf = smem + wave * B::kBytes;

    // copy offsets: 8 rows x 128 B per instruction, chunks swizzled by the row
    const uint32_t r8 = lane >> 3, c8 = lane & 7;
    const uint32_t row_off = r8 * (uint32_t)k + ((c8 ^ r8) << 4);
    const uint32_t q4_off = r8 * (uint32_t)(k >> 1) + ((c8 ^ r8) << 4);   // Q4_0: 128 bytes per row and step
    // operand reads: 8 bytes [32b + 8kq, +8) of a row = half b/4, chunk 2(b%4) + kq/2, byte 8(kq%2);
    // Q4_0 weights: chunk b, bytes 8(kq%2) .. +8, low nibbles for kq < 2, high nibbles above
    const uint32_t w4_col = (r >> 3) * 1024u + (r & 7) * 128u + (kq & 1) * 8u, w4_shift = 4 * (kq >> 1);
    uint32_t w_col[4], a_col[NT][4];
    uint32_t s_col[NT];
#pragma unroll
    for (uint32_t c = 0; c < 4; c++) w_col[c] = (r >> 3) * 2048u + (r & 7) * 128u + (((2 * c + (kq >> 1)) ^ (r & 7)) << 4) + (kq & 1) * 8u;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const uint32_t row = t * 16 + r < 8u * RT ? t * 16 + r : 8u * RT - 1;
#pragma unroll
        for (uint32_t c = 0; c < 4; c++)
            a_col[t][c] = B::oAct + (row >> 3) * 2048u + (row & 7) * 128u + (((2 * c + (kq >> 1)) ^ (row & 7)) << 4) + (kq & 1) * 8u;
        s_col[t] = B::oD8 + scale_col<RT>(t, kq);
    }

    v4f out[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) out[t] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};

    for (int64_t g = wave; g < kg; g += NW) {
        float4 xf[DIRECT ? 8 * RT : 1];
        if constexpr (DIRECT) {
            load_direct_q8<RT>(x + m0 * k, m - m0, k, g, lane, xf);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (Q4) {
#pragma unroll
            for (int rg = 0; rg < 2; rg++) dma16(w.p0 + (n_tile + rg * 8) * (k >> 1) + g * 128, q4_off, buf + rg * 1024);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int rg = i >> 1, kh = i & 1;
                dma16(w.p0 + (n_tile + rg * 8) * k + g * 256 + kh * 128, row_off, buf + i * 1024);
            }
        }
        if constexpr (!DIRECT) {
#pragma unroll
        for (int i = 0; i < 2 * RT; i++) {
            const int rg = i >> 1, kh = i & 1;
            if (RT > 1 || (int64_t)r8 < m - m0)   // (few rows: the others' copies are most of the activations')
                dma16(a.qs + (m0 + rg * 8) * k + g * 256 + kh * 128, row_off, buf + B::oAct + i * 1024);
        }
        issue_scales<RT>(a, m0, g, buf + B::oD8, lane);
        }
        // the eight block scales of this lane's weight row
        const u32x4_a4 dwv = *(const u32x4_a4 *)(w.p1 + ((n_tile + r) * kb + g * 8) * 2);
        if constexpr (DIRECT) {
            __builtin_amdgcn_sched_barrier(0);
            quantize_direct_q8<DT, RT>(xf, a, m0, m - m0, k, g, lane, tile == 0, buf);
        }
        __builtin_amdgcn_s_waitcnt(0);   // everything above has landed

        const uint32_t dww[4] = {dwv.x, dwv.y, dwv.z, dwv.w};
        auto block = [&](int b) {
            const float dw = cq_h2f((uint16_t)(dww[b >> 1] >> (16 * (b & 1))));
            const long wv = weight_bytes<Q4>(buf, b, r, w4_col, w4_shift, w_col);
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const long av = *(const long *)(buf + a_col[t][b & 3] + (b >> 2) * 1024);
                const v4f da = *(const v4f *)(buf + s_col[t] + b * 32);
                const v4i acc = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, wv, (v4i){0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (DUMP) {
                        const int64_t orow = m0 + t * 16 + kq * 4 + i;
                        if (orow < m) dump.i[(orow * w.n + n_tile + r) * kb + g * 8 + b] = acc[i];
                    } else {
                        out[t][i] = __builtin_fmaf((float)acc[i] * dw, da[i], out[t][i]);
                    }
                }
            }
        };
        each_block(kb - g * 8, block);
    }
    if (DUMP) return;
    if constexpr (OFF) add_min32<NT>(w, a, n_tile, m0, m, wave, NW, lane, out);

    // ---- sum the waves' partial tiles in wave order
#pragma unroll
    for (int t = 0; t < NT; t++) *(v4f *)(buf + t * 1024 + lane * 16) = out[t];
    __syncthreads();
    if (wave < NT) {
        v4f s = *(const v4f *)(smem + wave * 1024 + lane * 16);
#pragma unroll
        for (int o = 1; o < NW; o++) {
            const v4f p = *(const v4f *)(smem + o * B::kBytes + wave * 1024 + lane * 16);
            s += p;
        }
        const int64_t col = n_tile + r;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int64_t row = m0 + wave * 16 + kq * 4 + i;
            if (row < m) y[row * w.n + col] = s[i];
        }
    }
}

template <int DT, int RT, bool DUMP, int NW = kWaves, bool OFF = false>
__global__ void __launch_bounds__(NW * 64) skinny_blk32_kernel(cq_weight w, cq_act_view a, int64_t m0, int64_t m, float *__restrict__ y,
                                                                cq_mfma_dump dump) {
    skinny_blk32_body<DT, RT, DUMP, false, NW, OFF>(w, a, blockIdx.x, m0 + blockIdx.y * (8 * RT), m, y, dump);   // (a group of rows for each y)
}

// Mixture-of-experts form of the two: blockIdx.y is a tile of up to 8 * RT routed rows and names its expert's weights, so
// that a projection of all experts is one launch, as in the grouped tile kernel (gemm.hip).
template <int DT, int RT>
__global__ void __launch_bounds__(kThreads) skinny_grouped_kernel(cq_group_args ga, cq_act_view a, float *__restrict__ y) {
    const int tile = blockIdx.y;
    const int64_t m0 = ga.row0[tile], end = ga.row_end[tile], m = m0 + 8 * RT < end ? m0 + 8 * RT : end;
    const cq_weight w = ga.w[ga.expert[tile]];
    const cq_mfma_dump none{nullptr, nullptr, 0};
    if constexpr (DT == CQ_DTYPE_Q8_0 || DT == CQ_DTYPE_Q4_0) skinny_blk32_body<DT, RT, false>(w, a, blockIdx.x, m0, m, y, none);
    else skinny_body<DT, RT, false>(w, a, blockIdx.x, m0, m, y, none);
}

// Two or three weights on the same rows (q, k, v; gate and up): their 16-row tiles one after the other.  A weight with few
// rows (1024: 64 workgroups) does not fill the machine by itself.
template <int DT, int RT, bool OFF>
__global__ void __launch_bounds__(kThreads) skinny_shared_kernel(MultiArgs ma, cq_act_view a, int64_t m) {
    const uint32_t t = blockIdx.x;
    const int i = t >= ma.first[2] ? 2 : t >= ma.first[1] ? 1 : 0;
    const cq_weight w = ma.w[i];
    const cq_mfma_dump none{nullptr, nullptr, 0};
    if constexpr (DT == CQ_DTYPE_Q8_0 || DT == CQ_DTYPE_Q4_0) skinny_blk32_body<DT, RT, false, false, kWaves, OFF>(w, a, t - ma.first[i], 0, m, ma.y[i], none);
    else skinny_body<DT, RT, false, false, kWaves, OFF>(w, a, t - ma.first[i], 0, m, ma.y[i], none);
}

// ------------------------------------------------------------ the rows quantized by the waves that contract them ----
// One launch for the whole call: no quantizer launch in front, whose start and end are most of a small call (2.5 us of host time and
// 2-3 us on the device).  A wave quantizes the rows' blocks that it contracts into its own buffer, so that no wave waits for
// another; every workgroup repeats that, about 130 instructions for four rows of a block of 256, which is why it is for few weight rows
// and few activation rows (cq_skinny_direct_takes).  The workgroups of tile 0 leave the quantized rows in the workspace too, where a quantizer
// launch would have put them.
template <int DT>
__global__ void __launch_bounds__(kThreads) skinny_direct_kernel(cq_weight w, cq_act_view a, const float *__restrict__ x, int64_t m, float *__restrict__ y) {
    const cq_mfma_dump none{nullptr, nullptr, 0};
    const int64_t m0 = blockIdx.y * 8, end = m0 + 8 < m ? m0 + 8 : m;   // (the result tile has sixteen rows)
    if constexpr (DT == CQ_DTYPE_Q8_0 || DT == CQ_DTYPE_Q4_0) skinny_blk32_body<DT, 1, false, true>(w, a, blockIdx.x, m0, end, y, none, x);
    else skinny_body<DT, 1, false, true>(w, a, blockIdx.x, m0, end, y, none, x);
}

// ------------------------------------------- the same with everything of a workgroup in flight at once ----
// The kernel above has one 256-element step per wave in flight and spends most of its life waiting (56 % at
// s_waitcnt, the vector units 18 % busy).  Where every workgroup has one 16-row weight tile (n <= 16 x the number of
// compute units) and the call's quantized rows fit the LDS beside the weights, every wave requests all it will need -
// the activation slices, scales and weights of the K groups it owns (wave w: groups w, w + kWaves, ...) - right away,
// a single memory round trip, and the arithmetic follows as the data lands.
//   per K group g : act [RT][2 K-halves][8 rows][8 chunks], swizzled as above | d8 [RT row groups][8 blocks][8 rows] f32
//   then, per group: the 16 weight rows (Q8_0 4 KiB, Q4_0 2 KiB); a wave's first weight buffer also carries its
//                   partial results (1 KiB per 16 activation rows)
template <int DT, int RT> struct ResQ8 {
    static constexpr bool Q4 = DT == CQ_DTYPE_Q4_0;
    static constexpr int kWgt = Q4 ? 2048 : 4096;
    static constexpr int oD = RT * 2048, kActGrp = oD + RT * 256;
    static size_t bytes(int64_t kg) { return (size_t)kg * (kActGrp + kWgt); }
};

// m <= 8 * RT rows; n >= 16, one 16-row tile per workgroup; at most kMaxBpw K groups per wave.
template <int DT, int RT, int kWaves, bool DUMP, bool OFF = false>
__global__ void __launch_bounds__(kWaves * 64) skinny_blk32_resident_kernel(cq_weight w, cq_act_view a, int64_t m,
                                                                            float *__restrict__ y, cq_mfma_dump dump) {
    typedef ResQ8<DT, RT> R;
    constexpr bool Q4 = R::Q4;
    constexpr int NT = (RT + 1) / 2;   // 16-row tiles
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r = lane & 15, kq = lane >> 4;
    const int64_t k = w.k, kg = (w.k + 255) >> 8, kb = w.k >> 5;
    const int64_t n_tile = tile_row(blockIdx.x, w.n);
    uint8_t *wgt_base = smem + kg * R::kActGrp;

    const uint32_t r8 = lane >> 3, c8 = lane & 7;
    const uint32_t row_off = r8 * (uint32_t)k + ((c8 ^ r8) << 4);
    const uint32_t q4_off = r8 * (uint32_t)(k >> 1) + ((c8 ^ r8) << 4);
    const uint32_t w4_col = (r >> 3) * 1024u + (r & 7) * 128u + (kq & 1) * 8u, w4_shift = 4 * (kq >> 1);
    uint32_t w_col[4], a_col[NT][4];
#pragma unroll
    for (uint32_t c = 0; c < 4; c++) w_col[c] = (r >> 3) * 2048u + (r & 7) * 128u + (((2 * c + (kq >> 1)) ^ (r & 7)) << 4) + (kq & 1) * 8u;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const uint32_t row = t * 16 + r < 8u * RT ? t * 16 + r : 8u * RT - 1;
#pragma unroll
        for (uint32_t c = 0; c < 4; c++)
            a_col[t][c] = (row >> 3) * 2048u + (row & 7) * 128u + (((2 * c + (kq >> 1)) ^ (row & 7)) << 4) + (kq & 1) * 8u;
    }

    // ---- everything this wave will need, requested at once
    u32x4_a4 dwv[kMaxBpw];
#pragma unroll
    for (int j = 0; j < kMaxBpw; j++) {
        const int64_t g = wave + (int64_t)j * kWaves;
        if (g < kg) dwv[j] = *(const u32x4_a4 *)(w.p1 + ((n_tile + r) * kb + g * 8) * 2);
    }
#pragma unroll
    for (int j = 0; j < kMaxBpw; j++) {
        const int64_t g = wave + (int64_t)j * kWaves;
        if (g < kg) {
            uint8_t *act = smem + g * R::kActGrp, *wl = wgt_base + g * R::kWgt;
#pragma unroll
            for (int i = 0; i < 2 * RT; i++) {
                const int rg = i >> 1, kh = i & 1;
                dma16(a.qs + (int64_t)(rg * 8) * k + g * 256 + kh * 128, row_off, act + i * 1024);
            }
            issue_scales<RT>(a, 0, g, act + R::oD, lane);
            if (Q4) {
#pragma unroll
                for (int rg = 0; rg < 2; rg++) dma16(w.p0 + (n_tile + rg * 8) * (k >> 1) + g * 128, q4_off, wl + rg * 1024);
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int rg = i >> 1, kh = i & 1;
                    dma16(w.p0 + (n_tile + rg * 8) * k + g * 256 + kh * 128, row_off, wl + i * 1024);
                }
            }
        }
    }
    __builtin_amdgcn_s_waitcnt(0);   // everything above has landed

    v4f out[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) out[t] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < kMaxBpw; j++) {
        const int64_t g = wave + (int64_t)j * kWaves;
        if (g < kg) {
            const uint8_t *act = smem + g * R::kActGrp, *wl = wgt_base + g * R::kWgt;
            const uint32_t dww[4] = {dwv[j].x, dwv[j].y, dwv[j].z, dwv[j].w};
            auto block = [&](int b) {
                const float dw = cq_h2f((uint16_t)(dww[b >> 1] >> (16 * (b & 1))));
                const long wv = weight_bytes<Q4>(wl, b, r, w4_col, w4_shift, w_col);
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const long av = *(const long *)(act + a_col[t][b & 3] + (b >> 2) * 1024);
                    const v4f da = *(const v4f *)(act + R::oD + scale_col<RT>(t, kq) + b * 32);
                    const v4i acc = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, wv, (v4i){0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        if (DUMP) {
                            const int64_t orow = t * 16 + kq * 4 + i;
                            if (orow < m) dump.i[(orow * w.n + n_tile + r) * kb + g * 8 + b] = acc[i];
                        } else {
                            out[t][i] = __builtin_fmaf((float)acc[i] * dw, da[i], out[t][i]);
                        }
                    }
                }
            };
            each_block(kb - g * 8, block);
        }
    }
    if (DUMP) return;

    if constexpr (OFF) {
        if (wave < kg) add_min32<NT>(w, a, n_tile, 0, m, wave, kg < kWaves ? kg : kWaves, lane, out);
    }
    // ---- sum the waves' partial tiles in wave order (through each wave's first weight buffer)
    if (wave < kg) {
#pragma unroll
        for (int t = 0; t < NT; t++) *(v4f *)(wgt_base + (int64_t)wave * R::kWgt + t * 1024 + lane * 16) = out[t];
    }
    __syncthreads();
    if (wave < NT) {
        v4f s = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
        const int64_t nw = kg < kWaves ? kg : kWaves;   // waves that own a group
        for (int64_t o = 0; o < nw; o++) {
            const v4f p = *(const v4f *)(wgt_base + o * R::kWgt + wave * 1024 + lane * 16);
            s += p;
        }
        const int64_t col = n_tile + r;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int64_t row = wave * 16 + kq * 4 + i;
            if (row < m) y[row * w.n + col] = s[i];
        }
    }
}

// ------------------------------------- Q8_0 / Q4_0: resident activations, several tiles per workgroup ----
// The counterpart of skinny_resident_multi_kernel for the 32-element block types: one K group of 256 elements per wave
// (k <= 256 x waves), rounds of up to four 16-row tiles with one meeting per round, the weight scales through an LDS
// copy like the weights.  Q8_0 tiles are 4 KiB per wave and the LDS has room for one slot each: a tile's operands
// are read into registers first and the next tile's copies go out right behind them, under the MFMAs and the
// scaling.  Q4_0 (2 KiB) has two slots and keeps the tile after the next in flight.
//   LDS: activation groups as skinny_blk32_resident_kernel | per wave kSlots x {weights kWgt | scales 16 rows x 16 B};
//        the slots take the wave's partial results (1 KiB per tile) at the end of a round
template <int DT, int RT> struct ResQ8Multi {
    typedef ResQ8<DT, RT> R;
    static constexpr int kSlots = R::Q4 ? 2 : 1;
    static constexpr int oSc = R::kWgt, kSlot = R::kWgt + 256;
    static constexpr int kCopies = (R::Q4 ? 2 : 4) + 1;   // copy instructions per tile (blk32_multi_issue)
    static size_t bytes(int64_t kg) { return (size_t)kg * R::kActGrp + (size_t)kg * kSlots * kSlot; }
};

template <int DT, int RT>
__device__ __forceinline__ void blk32_multi_issue(uint8_t *__restrict__ slot, const cq_weight &w, int64_t n_tile, int64_t g, uint32_t row_off,
                                                  uint32_t q4_off, uint32_t ws_off, int lane) {
    typedef ResQ8Multi<DT, RT> M;
    const int64_t k = w.k, kb = w.k >> 5;
    if (M::R::Q4) {
#pragma unroll
        for (int rg = 0; rg < 2; rg++) dma16(w.p0 + (n_tile + rg * 8) * (k >> 1) + g * 128, q4_off, slot + rg * 1024);
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int rg = i >> 1, kh = i & 1;
            dma16(w.p0 + (n_tile + rg * 8) * k + g * 256 + kh * 128, row_off, slot + i * 1024);
        }
    }
    if (lane < 16) dma16(w.p1 + (n_tile * kb + g * 8) * 2, ws_off, slot + M::oSc);   // eight f16 scales of row `lane`
}

// One tile of one wave: operands out of `slot` into registers, the copies of a tile ahead into the free slot, MFMAs.
template <int DT, int RT, bool DUMP>
__device__ __forceinline__ void blk32_multi_step(uint8_t *__restrict__ slot, const uint8_t *__restrict__ act, int lane, const cq_weight &w,
                                                 bool ahead, int64_t rows_ahead, int64_t g, uint32_t row_off, uint32_t q4_off,
                                                 uint32_t ws_off, uint32_t w4_col, uint32_t w4_shift, const uint32_t (&w_col)[4],
                                                 const uint32_t (&a_col)[4], v4f &out, const cq_mfma_dump &dump, int64_t at, int64_t rs,
                                                 int64_t m) {
    typedef ResQ8Multi<DT, RT> M;
    typedef ResQ8<DT, RT> R;
    constexpr bool Q4 = R::Q4;
    const uint32_t r = lane & 15, kq = lane >> 4;
    const uint4 dwv = *(const uint4 *)(slot + M::oSc + r * 16u);
    long wv[8];
#pragma unroll
    for (int b = 0; b < 8; b++) {
        wv[b] = weight_bytes<Q4>(slot, b, r, w4_col, w4_shift, w_col);
    }
    if (ahead) {
        __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the reads above are done with the slot
        blk32_multi_issue<DT, RT>(slot, w, rows_ahead, g, row_off, q4_off, ws_off, lane);
    }
    const uint32_t dww[4] = {dwv.x, dwv.y, dwv.z, dwv.w};
    auto block = [&](int b) {
        const float dw = cq_h2f((uint16_t)(dww[b >> 1] >> (16 * (b & 1))));
        const long av = *(const long *)(act + a_col[b & 3] + (b >> 2) * 1024);
        const v4f da = *(const v4f *)(act + R::oD + scale_col<RT>(0, kq) + b * 32);
        const v4i acc = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, wv[b], (v4i){0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (DUMP) {
                const int64_t orow = kq * 4 + i;
                if (orow < m) dump.i[at + orow * rs + b] = acc[i];
            } else {
                out[i] = __builtin_fmaf((float)acc[i] * dw, da[i], out[i]);
            }
        }
    };
    each_block((w.k >> 5) - g * 8, block);
}

// m <= 8 * RT <= 16 rows; n >= 16; k / 256 <= kWaves.
template <int DT, int RT, int kWaves, bool DUMP>
__global__ void __launch_bounds__(kWaves * 64) skinny_blk32_multi_kernel(cq_weight w, cq_act_view a, int64_t m,
                                                                         float *__restrict__ y, cq_mfma_dump dump) {
    typedef ResQ8<DT, RT> R;
    typedef ResQ8Multi<DT, RT> M;
    constexpr bool Q4 = R::Q4;
    static_assert(RT <= 2, "one 16-row tile of activation rows");
    static_assert(M::kSlots * M::kSlot >= kTilesPerRound * 1024, "a round's partial tiles fit the wave's slots");
    constexpr int kAhead = 0x0F70 | M::kCopies;   // s_waitcnt vmcnt(copies of one tile)
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r = lane & 15, kq = lane >> 4;
    const int64_t k = w.k, kg = (w.k + 255) >> 8, kb = w.k >> 5;
    const int64_t tiles = (w.n + 15) / 16, G = gridDim.x;
    uint8_t *wgt_base = smem + kg * R::kActGrp;
    const bool has = wave < kg;   // this wave owns K group `wave`
    const int64_t g = wave;

    const uint32_t r8 = lane >> 3, c8 = lane & 7;
    const uint32_t row_off = r8 * (uint32_t)k + ((c8 ^ r8) << 4);
    const uint32_t q4_off = r8 * (uint32_t)(k >> 1) + ((c8 ^ r8) << 4);
    const uint32_t ws_off = (uint32_t)lane * (uint32_t)kb * 2u;   // lanes 0..15: the scales of row `lane`
    const uint32_t w4_col = (r >> 3) * 1024u + (r & 7) * 128u + (kq & 1) * 8u, w4_shift = 4 * (kq >> 1);
    uint32_t w_col[4], a_col[4];
    {
        const uint32_t row = r < 8u * RT ? r : 8u * RT - 1;
#pragma unroll
        for (uint32_t c = 0; c < 4; c++) {
            w_col[c] = (r >> 3) * 2048u + (r & 7) * 128u + (((2 * c + (kq >> 1)) ^ (r & 7)) << 4) + (kq & 1) * 8u;
            a_col[c] = (row >> 3) * 2048u + (row & 7) * 128u + (((2 * c + (kq >> 1)) ^ (row & 7)) << 4) + (kq & 1) * 8u;
        }
    }
    uint8_t *act = smem + g * R::kActGrp;
    uint8_t *ring = wgt_base + (size_t)g * M::kSlots * M::kSlot;

    // ---- the wave's activation group, once
    if (has) {
#pragma unroll
        for (int i = 0; i < 2 * RT; i++) {
            const int rg = i >> 1, kh = i & 1;
            dma16(a.qs + (int64_t)(rg * 8) * k + g * 256 + kh * 128, row_off, act + i * 1024);
        }
        issue_scales<RT>(a, 0, g, act + R::oD, lane);
    }
    for (int64_t t0 = blockIdx.x; t0 < tiles; t0 += kTilesPerRound * G) {
        int cnt = (int)((tiles - t0 + G - 1) / G);
        cnt = cnt < kTilesPerRound ? cnt : kTilesPerRound;
        if (has) {
            v4f o0 = {0.0f, 0.0f, 0.0f, 0.0f}, o1 = o0, o2 = o0, o3 = o0;
            blk32_multi_issue<DT, RT>(ring, w, tile_row(t0, w.n), g, row_off, q4_off, ws_off, lane);
            if (M::kSlots == 2 && cnt > 1) blk32_multi_issue<DT, RT>(ring + M::kSlot, w, tile_row(t0 + G, w.n), g, row_off, q4_off, ws_off, lane);
#pragma nounroll
            for (int i = 0; i < cnt; i++) {
                // everything but the copies of a tile in flight ahead has landed
                if (M::kSlots == 2 && i + 1 < cnt) __builtin_amdgcn_s_waitcnt(kAhead);
                else __builtin_amdgcn_s_waitcnt(0x0F70);
                const int64_t tile = t0 + i * G;
                v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
                blk32_multi_step<DT, RT, DUMP>(ring + (M::kSlots == 2 ? (i & 1) * M::kSlot : 0), act, lane, w, i + M::kSlots < cnt,
                                               tile_row(tile + M::kSlots * G, w.n), g, row_off, q4_off, ws_off, w4_col, w4_shift, w_col, a_col, acc, dump,
                                               (tile_row(tile, w.n) + r) * kb + g * 8, w.n * kb, m);
                if (i == 0) { o0 = acc; asm volatile(""); }
                else if (i == 1) { o1 = acc; asm volatile(""); }
                else if (i == 2) { o2 = acc; asm volatile(""); }
                else { o3 = acc; asm volatile(""); }
            }
            *(v4f *)(ring + lane * 16) = o0;
            *(v4f *)(ring + 1024 + lane * 16) = o1;
            *(v4f *)(ring + 2048 + lane * 16) = o2;
            *(v4f *)(ring + 3072 + lane * 16) = o3;
        }
        __syncthreads();
        if (wave < cnt && !DUMP) {   // wave i sums tile i of the round, in wave order
            v4f s = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
            const int64_t nw = kg < kWaves ? kg : kWaves;   // waves that own a group
            for (int64_t o = 0; o < nw; o++) {
                const v4f p = *(const v4f *)(wgt_base + (size_t)o * M::kSlots * M::kSlot + wave * 1024 + lane * 16);
                s += p;
            }
            const int64_t col = tile_row(t0 + wave * G, w.n) + r;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int64_t row = kq * 4 + i;
                if (row < m) y[row * w.n + col] = s[i];
            }
        }
        if (t0 + kTilesPerRound * G < tiles) __syncthreads();   // the sums have been read: the slots take the next round's copies
    }
}

// Weight types held in DT's planes that have an offset term.
template <int DT, bool DUMP> constexpr bool kCanOffset = !DUMP && (DT == CQ_DTYPE_Q8_0 || DT == CQ_DTYPE_Q6K);
bool has_offset(const cq_weight &w) { return cq_has_min32(w.ggml_dtype) || cq_has_min16(w.ggml_dtype); }

template <int DT, int RT, int NW, bool DUMP>
hipError_t launch_blk32_multi_inst(const cq_weight *w, cq_act_view a, int64_t m, float *y, size_t lds, unsigned grid, cq_mfma_dump d,
                                   hipStream_t s) {
    if (hipError_t e = cq_ensure_lds<skinny_blk32_multi_kernel<DT, RT, NW, DUMP>>(w->dev, lds); e != hipSuccess) return e;
    CQ_LAUNCH((skinny_blk32_multi_kernel<DT, RT, NW, DUMP>), grid, NW * 64, lds, s, *w, a, m, y, d);
    return hipGetLastError();
}

template <int DT, int RT, int NW, bool DUMP, bool OFF = false>
hipError_t launch_blk32_res_inst(const cq_weight *w, cq_act_view a, int64_t m, float *y, size_t lds, cq_mfma_dump d, hipStream_t s) {
    if (hipError_t e = cq_ensure_lds<skinny_blk32_resident_kernel<DT, RT, NW, DUMP, OFF>>(w->dev, lds); e != hipSuccess) return e;
    CQ_LAUNCH((skinny_blk32_resident_kernel<DT, RT, NW, DUMP, OFF>), (unsigned)((w->n + 15) / 16), NW * 64, lds, s, *w, a, m, y, d);
    return hipGetLastError();
}
// Takes the launch (true) where the resident kernel applies: one tile per workgroup, all operands in the LDS.
template <int DT, int RT, bool DUMP>
bool launch_blk32_res_rt(const cq_weight *w, cq_act_view a, int64_t m, float *y, cq_mfma_dump d, hipStream_t s, hipError_t *err) {
    const int64_t kg = (w->k + 255) >> 8, tiles = (w->n + 15) / 16;
    const int cus = cq_num_cus();
    const bool sixteen = kg > 8;
    if (tiles > cus) {
        // several tiles per workgroup: rounds of tiles with one meeting each, where a wave has one K group
        // (the types with an offset term: tile by tile, where it is added)
        if constexpr (RT <= 2) {
            const size_t lm = ResQ8Multi<DT, RT>::bytes(kg);
            if (!cq_has_min32(w->ggml_dtype) && sixteen && kg <= 16 && lm <= (size_t)kMaxLds && (uint64_t)w->n * (uint64_t)w->k < (1ull << 32)) {
                *err = launch_blk32_multi_inst<DT, RT, 16, DUMP>(w, a, m, y, lm, (unsigned)cus, d, s);
                return true;
            }
        }
        return false;
    }
    if (kg > (sixteen ? 16 : 8) * kMaxBpw) return false;
    if (RT > 2 && !sixteen) return false;   // (these go in groups of rows: cq_skinny_in_groups)
    constexpr int kFew = RT > 2 ? 16 : 8;
    const size_t lds = ResQ8<DT, RT>::bytes(kg);
    if (lds > (size_t)kMaxLds) return false;
    if constexpr (kCanOffset<DT, DUMP>) {
        if (has_offset(*w)) {
            *err = sixteen ? launch_blk32_res_inst<DT, RT, 16, DUMP, true>(w, a, m, y, lds, d, s) : launch_blk32_res_inst<DT, RT, kFew, DUMP, true>(w, a, m, y, lds, d, s);
            return true;
        }
    }
    *err = sixteen ? launch_blk32_res_inst<DT, RT, 16, DUMP>(w, a, m, y, lds, d, s) : launch_blk32_res_inst<DT, RT, kFew, DUMP>(w, a, m, y, lds, d, s);
    return true;
}
template <int DT, bool DUMP>
bool launch_blk32_res(const cq_weight *w, cq_act_view a, int64_t m, float *y, cq_mfma_dump d, hipStream_t s, hipError_t *err) {
    if (m <= 8) return launch_blk32_res_rt<DT, 1, DUMP>(w, a, m, y, d, s, err);
    if (m <= 16) return launch_blk32_res_rt<DT, 2, DUMP>(w, a, m, y, d, s, err);
    if (m <= 24) return launch_blk32_res_rt<DT, 3, DUMP>(w, a, m, y, d, s, err);
    if (m <= 32) return launch_blk32_res_rt<DT, 4, DUMP>(w, a, m, y, d, s, err);
    return false;
}

// DUMP (all launchers below): the launch cq_launch_skinny would make, storing the block integers through `d`.

// Sixteen waves to a workgroup instead of eight, for rows too long for the resident kernels: with a workgroup or less a CU, eight waves with a
// block each in flight leave the memory idle.  Measured, whole calls in us, eight waves -> sixteen, 4 and 8 rows: 4096 x 14336 Q4K 15.2 -> 13.6
// and 15.4 -> 14.6, Q4_0 16.0 -> 13.0 and 16.2 -> 13.8, Q6K 17.3 -> 16.2 and 17.5 -> 17.3; 2048 x 11008 Q4K 12.2 -> 10.7, Q4_0 13.2 -> 10.6.  Not
// for Q8_0, whose blocks are twice as long (4096 x 14336 18.1 -> 18.6), from nine rows on (Q4K 16.2 -> 17.3), or with more workgroups than CUs
// (8192 x 8192 Q6K 18.9 -> 20.9, Q5K 18.6 -> 20.6, Q4_0 14.8 -> 15.8), but for Q4K, of whose blocks two workgroups of sixteen waves fit a CU (8192 x
// 8192 16.0 -> 15.2, 5120 x 13824 18.4 -> 18.0; 14336 + 14336 x 4096 22.4 -> 25.2).
template <int DT, int RT> bool sixteen_waves(const cq_weight *w) {
    return RT == 1 && DT != CQ_DTYPE_Q8_0 && w->k > 16 * QK_K && (w->n + 15) / 16 <= (DT == CQ_DTYPE_Q4K ? 2 : 1) * cq_num_cus();
}

template <int DT, int RT, bool DUMP, int NW, bool OFF>
hipError_t launch_blk32_waves(const cq_weight *w, cq_act_view a, int64_t m0, int64_t m, float *y, cq_mfma_dump d, hipStream_t s, unsigned groups = 1) {
    const size_t lds = (size_t)BufQ8<DT, RT>::kBytes * NW;
    if (hipError_t e = cq_ensure_lds<skinny_blk32_kernel<DT, RT, DUMP, NW, OFF>>(w->dev, lds); e != hipSuccess) return e;
    CQ_LAUNCH((skinny_blk32_kernel<DT, RT, DUMP, NW, OFF>), dim3((unsigned)((w->n + 15) / 16), groups), NW * 64, lds, s, *w, a, m0, m, y, d);
    return hipGetLastError();
}
template <int DT, int RT, bool DUMP>
hipError_t launch_blk32_rt(const cq_weight *w, cq_act_view a, int64_t m, float *y, cq_mfma_dump d, hipStream_t s) {
    const bool sixteen = sixteen_waves<DT, RT>(w);
    constexpr int kMany = RT == 1 && DT != CQ_DTYPE_Q8_0 ? 16 : kWaves;
    if constexpr (kCanOffset<DT, DUMP>)
        if (has_offset(*w)) return sixteen ? launch_blk32_waves<DT, RT, DUMP, kMany, true>(w, a, 0, m, y, d, s) : launch_blk32_waves<DT, RT, DUMP, kWaves, true>(w, a, 0, m, y, d, s);
    return sixteen ? launch_blk32_waves<DT, RT, DUMP, kMany, false>(w, a, 0, m, y, d, s) : launch_blk32_waves<DT, RT, DUMP, kWaves, false>(w, a, 0, m, y, d, s);
}

// (up to 32 rows: more go in groups)
template <int DT, bool DUMP>
hipError_t launch_blk32(const cq_weight *w, cq_act_view a, int64_t m, float *y, cq_mfma_dump d, hipStream_t s) {
    if (m <= 8) return launch_blk32_rt<DT, 1, DUMP>(w, a, m, y, d, s);
    if (m <= 16) return launch_blk32_rt<DT, 2, DUMP>(w, a, m, y, d, s);
    if (m <= 24) return launch_blk32_rt<DT, 3, DUMP>(w, a, m, y, d, s);
    return launch_blk32_rt<DT, 4, DUMP>(w, a, m, y, d, s);
}

template <int DT, int RT, bool DUMP, int NW, bool OFF>
hipError_t launch_waves(const cq_weight *w, cq_act_view a, int64_t m0, int64_t m, float *y, cq_mfma_dump d, hipStream_t s, unsigned groups = 1) {
    const size_t lds = (size_t)Buf<DT, RT>::kBytes * NW;
    if (hipError_t e = cq_ensure_lds<skinny_kernel<DT, RT, DUMP, NW, OFF>>(w->dev, lds); e != hipSuccess) return e;
    CQ_LAUNCH((skinny_kernel<DT, RT, DUMP, NW, OFF>), dim3((unsigned)((w->n + 15) / 16), groups), NW * 64, lds, s, *w, a, m0, m, y, d);
    return hipGetLastError();
}
template <int DT, int RT, bool DUMP>
hipError_t launch_rt(const cq_weight *w, cq_act_view a, int64_t m, float *y, cq_mfma_dump d, hipStream_t s) {
    const bool sixteen = sixteen_waves<DT, RT>(w);
    constexpr int kMany = RT == 1 && DT != CQ_DTYPE_Q8_0 ? 16 : kWaves;
    if constexpr (kCanOffset<DT, DUMP>)
        if (has_offset(*w)) return sixteen ? launch_waves<DT, RT, DUMP, kMany, true>(w, a, 0, m, y, d, s) : launch_waves<DT, RT, DUMP, kWaves, true>(w, a, 0, m, y, d, s);
    return sixteen ? launch_waves<DT, RT, DUMP, kMany, false>(w, a, 0, m, y, d, s) : launch_waves<DT, RT, DUMP, kWaves, false>(w, a, 0, m, y, d, s);
}

// (up to 32 rows: more go in groups)
template <int DT, bool DUMP>
hipError_t launch_dt(const cq_weight *w, cq_act_view a, int64_t m, float *y, cq_mfma_dump d, hipStream_t s) {
    if (m <= 8) return launch_rt<DT, 1, DUMP>(w, a, m, y, d, s);
    if (m <= 16) return launch_rt<DT, 2, DUMP>(w, a, m, y, d, s);
    if (m <= 24) return launch_rt<DT, 3, DUMP>(w, a, m, y, d, s);
    return launch_rt<DT, 4, DUMP>(w, a, m, y, d, s);
}


// The resident-activation kernel where the call's activations and the weight buffers fit the LDS (see above).
template <int DT, int RT, int NW, bool DUMP, bool OFF = false>
hipError_t launch_res_inst(const cq_weight *w, cq_act_view a, int64_t m, float *y, size_t lds, cq_mfma_dump d, hipStream_t s) {
    if (hipError_t e = cq_ensure_lds<skinny_resident_kernel<DT, RT, NW, DUMP, OFF>>(w->dev, lds); e != hipSuccess) return e;
    CQ_LAUNCH((skinny_resident_kernel<DT, RT, NW, DUMP, OFF>), (unsigned)((w->n + 15) / 16), NW * 64, lds, s, *w, a, m, y, d);
    return hipGetLastError();
}
template <int DT, int RT, int NW, bool DUMP>
hipError_t launch_multi_inst(const cq_weight *w, cq_act_view a, int64_t m, float *y, size_t lds, unsigned grid, cq_mfma_dump d,
                             hipStream_t s) {
    if (hipError_t e = cq_ensure_lds<skinny_resident_multi_kernel<DT, RT, NW, DUMP>>(w->dev, lds); e != hipSuccess) return e;
    CQ_LAUNCH((skinny_resident_multi_kernel<DT, RT, NW, DUMP>), grid, NW * 64, lds, s, *w, a, m, y, d);
    return hipGetLastError();
}
template <int DT, int RT, bool DUMP>
bool launch_res_rt(const cq_weight *w, cq_act_view a, int64_t m, float *y, cq_mfma_dump d, hipStream_t s, hipError_t *err) {
    const int64_t kb = w->k >> 8, tiles = (w->n + 15) / 16;
    const int cus = cq_num_cus();
    const unsigned grid = (unsigned)(tiles < cus ? tiles : cus);
    const bool sixteen = kb > 8;
    if (kb > (sixteen ? 16 : 8) * kMaxBpw) return false;
    // the copies address every plane with 32-bit byte offsets
    if ((uint64_t)w->n * (uint64_t)kb * 128u >= (1ull << 32) || (uint64_t)a.m_stride * (uint64_t)w->k >= (1ull << 32)) return false;
    // Measured (Q4K, 16 rows, matmul kernel alone): 4096 x 4096, one tile per workgroup, 5.95 us against 6.5 us for the
    // kernel that copies activations per block; 11008 x 4096, two or three tiles per workgroup, 12.7 against 12.5 us
    // (also with the next tile's weights copied ahead into a second buffer): taken where every workgroup has one tile.
    if (tiles > grid) {
        // several tiles per workgroup: the kernel that meets once per round of tiles, where a wave has one K block
        if constexpr (RT <= 2 && (DT == CQ_DTYPE_Q4K || DT == CQ_DTYPE_Q5K)) {
            const size_t two = ResMulti<DT, RT>::bytes(kb);
            // Measured (Q4K, whole calls in us, the kernel that copies activations per block -> this one): 16 rows 11008 x 4096
            // 13.6 -> 12.6, 14336 x 4096 15.9 -> 14.3, 32000 x 4096 28.3 -> 24.1; 8 rows 11.7 -> 12.2, 14.1 -> 13.6, 24.1 -> 23.6:
            // with up to 8 rows five of the other kernel's workgroups share a CU and hide each other's waits.
            // K = 2048 (eight waves): 16 rows 8192 x 2048 10.0 -> 10.2; left with the other kernel.
            const bool pays = RT == 2 || tiles > 3 * (int64_t)cus;
            if (pays && sixteen && kb <= 16 && two <= (size_t)kMaxLds) {
                *err = launch_multi_inst<DT, RT, 16, DUMP>(w, a, m, y, two, grid, d, s);
                return true;
            }
        }
        return false;
    }
    const size_t one = Res<DT, RT>::bytes(kb);
    if (one <= (size_t)kMaxLds) {
        if constexpr (kCanOffset<DT, DUMP>) {
            if (has_offset(*w)) {
                *err = sixteen ? launch_res_inst<DT, RT, 16, DUMP, true>(w, a, m, y, one, d, s)
                               : launch_res_inst<DT, RT, 8, DUMP, true>(w, a, m, y, one, d, s);
                return true;
            }
        }
        *err = sixteen ? launch_res_inst<DT, RT, 16, DUMP>(w, a, m, y, one, d, s)
                       : launch_res_inst<DT, RT, 8, DUMP>(w, a, m, y, one, d, s);
        return true;
    }
    return false;
}
template <int DT, bool DUMP>
bool launch_res(const cq_weight *w, cq_act_view a, int64_t m, float *y, cq_mfma_dump d, hipStream_t s, hipError_t *err) {
    if (m <= 8) return launch_res_rt<DT, 1, DUMP>(w, a, m, y, d, s, err);
    if (m <= 16) return launch_res_rt<DT, 2, DUMP>(w, a, m, y, d, s, err);
    if (m <= 24) return launch_res_rt<DT, 3, DUMP>(w, a, m, y, d, s, err);
    if (m <= 32) return launch_res_rt<DT, 4, DUMP>(w, a, m, y, d, s, err);
    return false;
}

template <int DT, int RT, bool OFF>
hipError_t launch_shared_inst(const MultiArgs &ma, unsigned tiles, cq_act_view a, int64_t m, hipStream_t s) {
    const size_t lds = (size_t)(DT == CQ_DTYPE_Q8_0 || DT == CQ_DTYPE_Q4_0 ? (int)BufQ8<DT, RT>::kBytes : (int)Buf<DT, RT>::kBytes) * kWaves;
    if (hipError_t e = cq_ensure_lds<skinny_shared_kernel<DT, RT, OFF>>(ma.w[0].dev, lds); e != hipSuccess) return e;
    CQ_LAUNCH((skinny_shared_kernel<DT, RT, OFF>), tiles, kThreads, lds, s, ma, a, m);
    return hipGetLastError();
}
template <int DT, int RT>
hipError_t launch_shared_rt(const MultiArgs &ma, unsigned tiles, cq_act_view a, int64_t m, hipStream_t s) {
    if constexpr (kCanOffset<DT, false>)
        if (has_offset(ma.w[0])) return launch_shared_inst<DT, RT, true>(ma, tiles, a, m, s);   // (all of one type)
    return launch_shared_inst<DT, RT, false>(ma, tiles, a, m, s);
}
// Nine rows and more of Q4K with nine to sixteen blocks a row: by rounds of tiles over all the weights, as launch_res_rt does for one.  Measured
// with rms_norm in front, whole calls in us, tile by tile (for many rows a launch for each weight) -> rounds, 16 rows: 3 x 4096 x 4096 17.1 -> 15.1,
// 4096 + 1024 + 1024 x 4096 13.7 -> 12.2, 2 x 6912 x 2560 14.3 -> 13.9, 2 x 14336 x 4096 28.0 -> 27.9, 2 x 28672 40.0 -> 40.0.  Not with up to eight
// rows (3 x 4096 x 4096, 4 rows 14.3 -> 14.9, 2 x 14336 22.1 -> 24.2: more workgroups share a CU) and not for Q5K (16 rows, 2 x 14336 32.0 -> 32.0,
// 2 x 6912 x 2560 17.3 -> 17.5).
bool shared_by_rounds(const MultiArgs &ma, const cq_act_view &a, int64_t m) {
    const int64_t kb = ma.w[0].k >> 8;
    for (const cq_weight &w : ma.w)
        if ((uint64_t)w.n * (uint64_t)kb * 128u >= (1ull << 32)) return false;   // (32-bit byte offsets)
    return m > 8 && kb > 8 && kb <= 16 && ResMulti<CQ_DTYPE_Q4K, 2>::bytes(kb) <= (size_t)kMaxLds && (uint64_t)a.m_stride * (uint64_t)ma.w[0].k < (1ull << 32);
}
hipError_t launch_shared_rounds(const MultiArgs &ma, unsigned tiles, cq_act_view a, int64_t m, hipStream_t s) {
    const size_t lds = ResMulti<CQ_DTYPE_Q4K, 2>::bytes(ma.w[0].k >> 8);
    if (hipError_t e = cq_ensure_lds<skinny_shared_rounds_kernel>(ma.w[0].dev, lds); e != hipSuccess) return e;
    const unsigned cus = (unsigned)cq_num_cus();
    CQ_LAUNCH(skinny_shared_rounds_kernel, tiles < cus ? tiles : cus, 16 * 64, lds, s, ma, tiles, a, m);
    return hipGetLastError();
}
template <int DT> hipError_t launch_shared(const MultiArgs &ma, unsigned tiles, cq_act_view a, int64_t m, hipStream_t s) {
    if (DT == CQ_DTYPE_Q4K && shared_by_rounds(ma, a, m)) return launch_shared_rounds(ma, tiles, a, m, s);
    return m <= 8 ? launch_shared_rt<DT, 1>(ma, tiles, a, m, s) : launch_shared_rt<DT, 2>(ma, tiles, a, m, s);
}

template <int DT, int RT>
hipError_t launch_grouped_rt(const cq_weight *const *experts, int n_experts, const int32_t *offsets, cq_act_view a, float *y, hipStream_t s) {
    cq_group_args ga;
    const int tiles = cq_group_table(experts, n_experts, offsets, 8 * RT, &ga);
    if (tiles <= 0) return tiles == 0 ? hipSuccess : hipErrorInvalidConfiguration;
    const size_t lds = (size_t)(DT == CQ_DTYPE_Q8_0 || DT == CQ_DTYPE_Q4_0 ? (int)BufQ8<DT, RT>::kBytes : (int)Buf<DT, RT>::kBytes) * kWaves;
    if (hipError_t e = cq_ensure_lds<skinny_grouped_kernel<DT, RT>>(experts[0]->dev, lds); e != hipSuccess) return e;
    CQ_LAUNCH((skinny_grouped_kernel<DT, RT>), dim3((unsigned)((experts[0]->n + 15) / 16), (unsigned)tiles), kThreads, lds, s, ga, a, y);
    return hipGetLastError();
}
// Groups of eight rows a tile, and the us of the launch with its quantizer: weight bytes of the experts that have rows, blocks of all tiles per CU
// and bytes stored.  Up to 16 rows for the fullest expert what holds them (Q8_0 beyond eight: by the estimate), beyond by the estimate among 16 and
// 24 (Q8_0 8 and 16, Q4_0 16); 32 only where more tiles than a launch names would be needed.  Fitted to 8600 grouped calls (8 experts, 1024
// to 4096 elements by 1.5 to 3.5 times as many, either way round, 2 to 512 routed rows), 5 to 8 % rms.
struct GroupedPlan {
    int rt;
    double us;
};
GroupedPlan plan_grouped(const cq_weight *w, int n_experts, const int32_t *offsets) {
    const int t = w->dtype == CQ_DTYPE_Q4K ? 0 : w->dtype == CQ_DTYPE_Q5K ? 1 : w->dtype == CQ_DTYPE_Q8_0 ? 3 : w->dtype == CQ_DTYPE_Q4_0 ? 4 : 2;
    static constexpr double bits[5] = {4.625, 5.625, 6.5625, 8.5, 4.5};
    static constexpr double bytes_us[3][5] = {{0.044, 0.056, 0.049, 0.068, 0.061}, {0.054, 0.074, 0.062, 0.068, 0.055}, {0.070, 0.066, 0.059, 0, 0}};
    static constexpr double block_us[3][5] = {{0.070, 0.108, 0.100, 0.085, 0.071}, {0.084, 0.101, 0.101, 0.108, 0.088}, {0.099, 0.129, 0.127, 0, 0}};
    static constexpr double out_us[3][5] = {{2.5, 3.8, 3.0, 2.5, 3.5}, {1.6, 3.5, 2.8, 2.3, 1.8}, {2.4, 2.8, 2.1, 0, 0}};
    int64_t most = 0, active = 0;
    for (int e = 0; e < n_experts; e++) {
        const int64_t rows = offsets[e + 1] - offsets[e];
        most = rows > most ? rows : most;
        active += rows > 0;
    }
    const int first = most <= 8 || t == 3 ? 1 : 2, last = most <= 8 ? 1 : most <= 16 || t >= 3 ? 2 : 3;
    const double mb = (double)active * (double)w->n * (double)w->k * bits[t] / 8e6, out = (double)w->n * (double)offsets[n_experts] * 4e-6;
    GroupedPlan best{4, 1e30};
    for (int rt = first; rt <= last; rt++) {
        const int64_t tiles = cq_group_tiles(offsets, n_experts, 8 * rt);
        if (tiles > kMaxGroupTiles) continue;
        const double blocks = (double)w->k / 256.0 * (double)((w->n + 15) / 16) * (double)tiles / (double)cq_num_cus();
        const double us = 7.0 + bytes_us[rt - 1][t] * mb + block_us[rt - 1][t] * blocks + out_us[rt - 1][t] * out;
        if (us < best.us) best = GroupedPlan{rt, us};
    }
    return best;
}
template <int DT>
hipError_t launch_grouped(const cq_weight *const *experts, int n_experts, const int32_t *offsets, cq_act_view a, float *y, hipStream_t s) {
    switch (plan_grouped(experts[0], n_experts, offsets).rt) {
    case 1: return launch_grouped_rt<DT, 1>(experts, n_experts, offsets, a, y, s);
    case 2: return launch_grouped_rt<DT, 2>(experts, n_experts, offsets, a, y, s);
    case 3:
        if constexpr (DT != CQ_DTYPE_Q8_0 && DT != CQ_DTYPE_Q4_0) return launch_grouped_rt<DT, 3>(experts, n_experts, offsets, a, y, s);
        return hipErrorInvalidValue;   // (never planned)
    default: return launch_grouped_rt<DT, 4>(experts, n_experts, offsets, a, y, s);
    }
}

// All the rows in one launch, 8 * RT of them to a workgroup.
template <int DT, int RT, bool DUMP, bool OFF>
hipError_t launch_groups_inst(const cq_weight *w, cq_act_view a, int64_t m0, int64_t m, float *y, cq_mfma_dump d, hipStream_t s, unsigned groups) {
    if constexpr (DT == CQ_DTYPE_Q8_0 || DT == CQ_DTYPE_Q4_0) return launch_blk32_waves<DT, RT, DUMP, kWaves, OFF>(w, a, m0, m, y, d, s, groups);
    else return launch_waves<DT, RT, DUMP, kWaves, OFF>(w, a, m0, m, y, d, s, groups);
}
template <int DT, int RT, bool DUMP>
hipError_t launch_groups(const cq_weight *w, cq_act_view a, int64_t m, float *y, cq_mfma_dump d, hipStream_t s) {
    const int64_t most = (int64_t)8 * RT * 65535;
    for (int64_t m0 = 0; m0 < m; m0 += most) {
        const unsigned groups = (unsigned)(((m - m0 < most ? m - m0 : most) + 8 * RT - 1) / (8 * RT));
        hipError_t e = hipErrorInvalidValue;
        if constexpr (kCanOffset<DT, DUMP>) e = has_offset(*w) ? launch_groups_inst<DT, RT, DUMP, true>(w, a, m0, m, y, d, s, groups)
                                                               : launch_groups_inst<DT, RT, DUMP, false>(w, a, m0, m, y, d, s, groups);
        else e = launch_groups_inst<DT, RT, DUMP, false>(w, a, m0, m, y, d, s, groups);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
// More than 16 rows, us beside the quantizer and the stores: groups of 16 and (K-quants) of 32 rows.  A workgroup goes through a row in steps of
// 2048 elements, 256 a wave; three or two of them share a CU with 16 rows, one with 32 (LDS; groups of 32 are never ahead for Q8_0 and Q4_0).
// Fitted to 35000 measured calls of Q4K, Q5K and Q6K and 21000 of Q8_0 and Q4_0 (24 to 9400 weight rows, k 256 to 15104, 17 to 1024 rows), 7 to 9 %
// rms.
struct GroupsUs {
    double sixteen, thirty_two;
};
GroupsUs groups_us(const cq_weight *w, int64_t m) {
    const double tiles = (double)((w->n + 15) / 16), cus = (double)cq_num_cus(), steps = (double)((w->k + 2047) / 2048);
    const double f16 = tiles * (double)((m + 15) / 16) / cus, f32 = tiles * (double)((m + 31) / 32) / cus, rounds = f32 <= 1.0 ? 1.0 : ceil(f32);
    if (w->dtype == CQ_DTYPE_Q8_0) return {5.0 + steps * (1.19 + 0.96 * f16), 1e30};
    if (w->dtype == CQ_DTYPE_Q4_0) return {5.15 + steps * (1.25 + 0.66 * f16), 1e30};
    const int t = w->dtype == CQ_DTYPE_Q4K ? 0 : w->dtype == CQ_DTYPE_Q5K ? 1 : 2;
    static constexpr double a16[3] = {0.94, 1.19, 1.05}, b16[3] = {0.62, 0.94, 0.88};
    static constexpr double a32[3] = {1.25, 1.65, 1.46}, b32[3] = {0.16, 0.22, 0.23}, c32[3] = {0.49, 0.32, 0.41};
    return {5.35 + steps * (a16[t] + b16[t] * f16), 5.15 + steps * (a32[t] * rounds + b32[t] * f32) + c32[t] * rounds};
}

template <int DT, bool DUMP>
hipError_t launch_in_groups(const cq_weight *w, cq_act_view a, int64_t m, float *y, cq_mfma_dump d, hipStream_t s) {
    const GroupsUs us = groups_us(w, m);
    if (us.sixteen <= us.thirty_two || m <= 32) return launch_groups<DT, 2, DUMP>(w, a, m, y, d, s);
    if constexpr (DT != CQ_DTYPE_Q8_0 && DT != CQ_DTYPE_Q4_0) return launch_groups<DT, 4, DUMP>(w, a, m, y, d, s);
    return hipErrorInvalidValue;
}

template <bool DUMP>
hipError_t launch_any(const cq_weight *w, cq_act_view a, int act_dtype, int64_t m, float *y, cq_mfma_dump d, hipStream_t s) {
    if (!cq_skinny_takes(w, act_dtype)) return hipErrorNotSupported;
    if (m == 0) return hipSuccess;
    if (a.m_stride < (m + 31) / 32 * 32) return hipErrorInvalidValue;   // whole 8-row groups are copied
    hipError_t e = hipSuccess;
    if (cq_skinny_in_groups(w, m)) {
        switch (w->dtype) {
        case CQ_DTYPE_Q8_0: return launch_in_groups<CQ_DTYPE_Q8_0, DUMP>(w, a, m, y, d, s);
        case CQ_DTYPE_Q4_0: return launch_in_groups<CQ_DTYPE_Q4_0, DUMP>(w, a, m, y, d, s);
        case CQ_DTYPE_Q4K: return launch_in_groups<CQ_DTYPE_Q4K, DUMP>(w, a, m, y, d, s);
        case CQ_DTYPE_Q5K: return launch_in_groups<CQ_DTYPE_Q5K, DUMP>(w, a, m, y, d, s);
        default: return launch_in_groups<CQ_DTYPE_Q6K, DUMP>(w, a, m, y, d, s);
        }
    }
    if (w->dtype == CQ_DTYPE_Q8_0 && launch_blk32_res<CQ_DTYPE_Q8_0, DUMP>(w, a, m, y, d, s, &e)) return e;
    if (w->dtype == CQ_DTYPE_Q4_0 && launch_blk32_res<CQ_DTYPE_Q4_0, DUMP>(w, a, m, y, d, s, &e)) return e;
    if (w->dtype == CQ_DTYPE_Q8_0) return launch_blk32<CQ_DTYPE_Q8_0, DUMP>(w, a, m, y, d, s);
    if (w->dtype == CQ_DTYPE_Q4_0) return launch_blk32<CQ_DTYPE_Q4_0, DUMP>(w, a, m, y, d, s);
    if (w->dtype == CQ_DTYPE_Q4K && launch_res<CQ_DTYPE_Q4K, DUMP>(w, a, m, y, d, s, &e)) return e;
    if (w->dtype == CQ_DTYPE_Q5K && launch_res<CQ_DTYPE_Q5K, DUMP>(w, a, m, y, d, s, &e)) return e;
    if (w->dtype == CQ_DTYPE_Q6K && launch_res<CQ_DTYPE_Q6K, DUMP>(w, a, m, y, d, s, &e)) return e;
    if (w->dtype == CQ_DTYPE_Q4K) return launch_dt<CQ_DTYPE_Q4K, DUMP>(w, a, m, y, d, s);
    if (w->dtype == CQ_DTYPE_Q5K) return launch_dt<CQ_DTYPE_Q5K, DUMP>(w, a, m, y, d, s);
    return launch_dt<CQ_DTYPE_Q6K, DUMP>(w, a, m, y, d, s);
}

template <int DT> hipError_t launch_direct(const cq_weight *w, cq_act_view a, const float *x, int64_t m, float *y, hipStream_t s) {
    const size_t lds = (size_t)(DT == CQ_DTYPE_Q8_0 || DT == CQ_DTYPE_Q4_0 ? (int)BufQ8<DT, 1>::kBytes : (int)Buf<DT, 1>::kBytes) * kWaves;
    if (hipError_t e = cq_ensure_lds<skinny_direct_kernel<DT>>(w->dev, lds); e != hipSuccess) return e;
    CQ_LAUNCH((skinny_direct_kernel<DT>), dim3((unsigned)((w->n + 15) / 16), (unsigned)((m + 7) / 8)), kThreads, lds, s, *w, a, x, m, y);
    return hipGetLastError();
}

}  // namespace

bool cq_skinny_takes(const cq_weight *w, int act_dtype) {
    // the copies address 8 rows of activations and 16 rows of a weight plane with 32-bit offsets
    const bool kquant = (w->dtype == CQ_DTYPE_Q4K || w->dtype == CQ_DTYPE_Q5K || w->dtype == CQ_DTYPE_Q6K) && act_dtype == CQ_DTYPE_Q8K;
    const bool q8 = (w->dtype == CQ_DTYPE_Q8_0 || w->dtype == CQ_DTYPE_Q4_0) && act_dtype == CQ_DTYPE_Q8_0 && w->k % 64 == 0;
    return (kquant || q8) && w->k >= 256 && w->k <= (1 << 24) && w->n >= 16;
}
// More than 16 rows in groups of 16 or 32, one launch: beyond 32 rows always (against a launch for every 32 rows), up to 32 where a group of 16 for
// every CU does it (K-quants: and a wave has more than one block; the resident kernel is as fast below.  Q8_0 / Q4_0 with one step: two
// groups for every CU).  Whole calls, us, before -> groups: Q4K 1024 x 4096 with 24 / 64 / 128 rows 9.4 -> 7.7 / 13.9 -> 8.3 / 14.0 -> 9.4, 411 x
// 3584 with 128 17.6 -> 8.6, Q6K 512 x 4096 with 33 13.4 -> 8.1, 2048 x 2048 with 64 11.7 -> 7.7, Q3K 256 x 13312 with 52 22.0 -> 13.9, Q8_0 1528 x 960
// with 48 11.3 -> 7.2; without a tile kernel Q4K 48 x 3072 with 256 rows 39 -> 8.2, Q8_0 28 x 1920 with 48 11.1 -> 6.8.
bool cq_skinny_in_groups(const cq_weight *w, int64_t m) {
    const bool blk32 = w->dtype == CQ_DTYPE_Q8_0 || w->dtype == CQ_DTYPE_Q4_0, one_step = w->k <= 8 * QK_K;
    const int64_t pairs = (w->n + 15) / 16 * 2, cus = cq_num_cus();   // groups of 16 with up to 32 rows
    return m > 32 || (m > 16 && (blk32 ? pairs <= (one_step ? 2 : 1) * cus : !one_step && pairs <= cus));
}
// (33 to 128 weight rows: 0.4 us more for every MiB of quantized rows.  With so few weight tiles the launch waits for the rows, and the tile kernel,
// half of whose waves are idle there, is ahead of its estimate.  Without that the choice lost up to a fifth, us, tiles -> groups: Q4K 128 x 8192
// with 2048 rows 32.6 -> 41.0, 96 x 8192 with 512 14.1 -> 16.8, Q8_0 96 x 4096 with 1024 15.5 -> 18.5.  Of 375 cases (64, 96 and 128 weight rows,
// 128 to 2048 rows) 76 change to the tiles: 53 are more than 3 % faster, 7 slower, by 7 % at most.)
double cq_skinny_groups_us(const cq_weight *w, int64_t m) {
    const GroupsUs us = groups_us(w, m);
    const double rows = w->n > 32 && w->n <= 128 ? 0.4 * (double)m * (double)w->k / (double)(1 << 20) : 0.0;
    return (us.sixteen < us.thirty_two ? us.sixteen : us.thirty_two) + rows;
}
bool cq_skinny_supported(const cq_weight *w, int act_dtype) {
    return cq_skinny_takes(w, act_dtype) && w->k % 256 == 0 && w->n % 16 == 0;
}

hipError_t cq_launch_skinny(const cq_weight *w, cq_act_view a, int act_dtype, int64_t m, float *y, hipStream_t s) {
    return launch_any<false>(w, a, act_dtype, m, y, cq_mfma_dump{nullptr, nullptr, 0}, s);
}

hipError_t cq_launch_skinny_dump(const cq_weight *w, cq_act_view a, int act_dtype, int64_t m, cq_mfma_dump d, hipStream_t s) {
    return launch_any<true>(w, a, act_dtype, m, nullptr, d, s);
}

// The rows quantized by the contracting waves (where the dot-product kernel does not take them in one launch): where the quantizing that
// every workgroup repeats for its eight rows costs less than the launch it saves.  Measured, us back to back / from a graph, against the two
// launches:
//   Q4K 1024 x 1024, 5 rows 4.8 / 4.5 against 7.5 / 5.0; 8 rows 4.8 / 4.5 against 7.4 / 5.1; 326 x 768, 12 rows 4.7 / 4.7 against 8.6 / 5.7; Q6K
//   4096 x 1024, 8 rows 5.0 / 4.7 against 7.3 / 5.3; Q8_0 1024 x 1024, 5 rows 5.0 / 4.8 against 8.0 / 5.2
// level or a little behind from a graph at the most rows of the 32-element types (Q8_0 1024 x 1024, 8 rows 5.9 / 5.6 against 7.9 / 5.3, Q4_0, 7
// rows 5.9 / 5.7 against 8.0 / 5.5), and beyond the limits below behind from a graph or everywhere: two blocks a wave or two workgroups a CU double the quantizing
// (Q4K 2048 x 2048, 8 rows 6.0 against 6.8 / 5.6; 8192 x 2048 10.6 against 7.3), Q4_0 with 8 rows 5.9 / 5.7 against 7.4 / 5.5.
// More than eight rows (K-quants): up to a workgroup a CU and a block a wave, on random shapes 1.25 to 1.7 times as fast back to back (1024 x 1024
// with 32 rows 8.1 -> 5.2, Q6K 512 x 2048 with 64 11.9 -> 6.8, Q5K 256 x 1024 with 128 11.3 -> 5.6) and at least 1.03 times from a graph; Q8_0 and
// Q4_0, whose rows a wave quantizes one by one, 1.05 to 1.4 but from a graph 0.8 to 0.95 (Q4_0 20 x 1536 with 28 rows 8.5 / 6.2 -> 7.2 / 7.5).
bool cq_skinny_direct_takes(const cq_weight *w, int act_dtype, int64_t m) {
    if (m < 2 || cq_has_min32(w->ggml_dtype) || cq_has_min16(w->ggml_dtype) || !cq_skinny_takes(w, act_dtype)) return false;
    const int64_t groups = (w->n + 15) / 16 * ((m + 7) / 8);
    if (m > 8) return act_dtype == CQ_DTYPE_Q8K && groups <= cq_num_cus() && w->k <= 8 * QK_K;
    return m <= (w->dtype == CQ_DTYPE_Q4_0 ? 7 : 8) && w->n <= 4096 && w->k <= (m <= 4 ? 2048 : 1024);
}
hipError_t cq_launch_skinny_direct(const cq_weight *w, cq_act_view a, const float *x, int64_t m, float *y, hipStream_t s) {
    switch (w->dtype) {
    case CQ_DTYPE_Q8_0: return launch_direct<CQ_DTYPE_Q8_0>(w, a, x, m, y, s);
    case CQ_DTYPE_Q4_0: return launch_direct<CQ_DTYPE_Q4_0>(w, a, x, m, y, s);
    case CQ_DTYPE_Q4K: return launch_direct<CQ_DTYPE_Q4K>(w, a, x, m, y, s);
    case CQ_DTYPE_Q5K: return launch_direct<CQ_DTYPE_Q5K>(w, a, x, m, y, s);
    default: return launch_direct<CQ_DTYPE_Q6K>(w, a, x, m, y, s);
    }
}

bool cq_skinny_grouped_takes(const cq_weight *const *experts, int n_experts, const int32_t *offsets, int act_dtype) {
    if (n_experts > kMaxGroupExperts || !cq_skinny_takes(experts[0], act_dtype)) return false;
    return cq_group_tiles(offsets, n_experts, 8 * plan_grouped(experts[0], n_experts, offsets).rt) <= kMaxGroupTiles;
}
double cq_skinny_grouped_us(const cq_weight *w, int n_experts, const int32_t *offsets) { return plan_grouped(w, n_experts, offsets).us; }

hipError_t cq_launch_skinny_grouped(const cq_weight *const *experts, int n_experts, const int32_t *offsets, cq_act_view a, float *y,
                                    hipStream_t s) {
    if (a.m_stride < (int64_t)offsets[n_experts] + 31) return hipErrorInvalidValue;   // tiles of up to 32 rows from any row on
    switch (experts[0]->dtype) {
    case CQ_DTYPE_Q8_0: return launch_grouped<CQ_DTYPE_Q8_0>(experts, n_experts, offsets, a, y, s);
    case CQ_DTYPE_Q4_0: return launch_grouped<CQ_DTYPE_Q4_0>(experts, n_experts, offsets, a, y, s);
    case CQ_DTYPE_Q4K: return launch_grouped<CQ_DTYPE_Q4K>(experts, n_experts, offsets, a, y, s);
    case CQ_DTYPE_Q5K: return launch_grouped<CQ_DTYPE_Q5K>(experts, n_experts, offsets, a, y, s);
    default: return launch_grouped<CQ_DTYPE_Q6K>(experts, n_experts, offsets, a, y, s);
    }
}

// 17 to 32 rows of a K-quant: whether the split-K kernel is ahead of the tiles (us of both whole calls, the quantizer in front of each; thousands of
// weight rows, K / 1024).  It walks K once for every round of sixteen weight rows a compute unit, which the bytes hide behind at first, and beyond 24
// rows one workgroup less fits a compute unit; the tiles cost by their plan, K split or not (cq_gemm_few_us).  Both fitted to 165 shapes of each
// type at 17, 24 and 32 rows, weights from HBM (8192 to 128256 weight rows with K 512 to 16384, 3072 to 7168 with K 6400 to 28672), mostly to those
// where the kernels are close: the choice is 0.3 % behind the better one on average, 10 % at worst and more than 3 % in 4 % of the calls; lines at
// 14336 weight rows (24 rows) and 12288 (32) are 4.6 % behind on average, 61 % at worst.  Some (us, split K / tiles): 24 rows Q4K 8192 x 14336
// 31.8/26.6, 4128 x 12288 25.6/19.8, 4096 x 14336 18.9/21.0, Q5K 16384 x 3072 19.7/23.8, 6144 x 16384 38.3/33.7; 32 rows Q4K 11008 x 8192 32.5/25.5,
// 10240 x 1024 11.6/9.9, 4096 x 14336 20.8/22.0, Q6K 8192 x 14336 41.1/34.7, 12288 x 3072 20.3/23.4.  Small weights, whose rows go in groups
// (cq_skinny_in_groups), stay: level, the tiles up to 18 % ahead only with K beyond 20000 (Q4K 1024 x 28672 23.5/20.2).
bool cq_skinny_few_ahead(const cq_weight *w, int64_t m) {
    if (cq_skinny_in_groups(w, m)) return true;
    static constexpr double split[2][3][4] = {{{6.14, 0.083, 0.030, 0.733}, {6.34, 0.131, 0.026, 0.884}, {6.32, 0.112, 0.044, 0.810}},
                                              {{5.22, 0.329, 0.014, 0.953}, {5.55, 0.408, 0.009, 1.085}, {5.55, 0.383, 0.033, 0.978}}};
    const double(&c)[4] = split[m > 24][w->dtype == CQ_DTYPE_Q4K ? 0 : w->dtype == CQ_DTYPE_Q5K ? 1 : 2];
    const int64_t cus = cq_num_cus(), rounds = ((w->n + 15) / 16 + cus - 1) / cus;
    const double rows = (double)w->n / 1000.0, k = (double)w->k / 1024.0;
    return c[0] + c[1] * rows + c[2] * rows * k + c[3] * k * (double)rounds < cq_gemm_few_us(w, m);
}

// One launch over all the weights rather than a launch each.  Measured with rms_norm in front, weights from HBM, five types, 2..16 rows,
// ten pairs and triples from 1024 to 28672 weight rows and K = 1024..8192 (us of the whole call, one launch / a launch each):
// the one launch is ahead everywhere (Q4K, 8 rows: 4096 + 1024 + 1024 x 4096 12.2 / 18.9, 2 x 14336 x 4096 24.3 / 26.8, 2 x 28672
// x 8192 77.5 / 82.7; 16 rows: Q6K 2 x 14336 x 4096 32.2 / 37.2, Q8_0 2 x 11008 x 4096 31.2 / 31.8).
bool cq_skinny_shared_takes(const cq_weight *const *ws, int count, int64_t m, int act_dtype) {
    if (count < 2 || count > kMultiMax || m > 16) return false;
    for (int i = 0; i < count; i++)
        if (!cq_skinny_takes(ws[i], act_dtype)) return false;
    return true;
}

hipError_t cq_launch_skinny_shared(const cq_weight *const *ws, int count, cq_act_view a, int64_t m, float *const *ys, hipStream_t s) {
    if (a.m_stride < (m + 31) / 32 * 32) return hipErrorInvalidValue;   // whole 8-row groups are copied
    MultiArgs ma;
    int64_t tiles = 0;
    for (int i = 0; i < kMultiMax; i++) {
        const int j = i < count ? i : count - 1;   // (an unused place repeats the last weight and begins past the last tile)
        ma.w[i] = *ws[j];
        ma.y[i] = ys[j];
        ma.first[i] = (uint32_t)tiles;
        if (i < count) tiles += (ws[i]->n + 15) / 16;
    }
    switch (ws[0]->dtype) {
    case CQ_DTYPE_Q8_0: return launch_shared<CQ_DTYPE_Q8_0>(ma, (unsigned)tiles, a, m, s);
    case CQ_DTYPE_Q4_0: return launch_shared<CQ_DTYPE_Q4_0>(ma, (unsigned)tiles, a, m, s);
    case CQ_DTYPE_Q4K: return launch_shared<CQ_DTYPE_Q4K>(ma, (unsigned)tiles, a, m, s);
    case CQ_DTYPE_Q5K: return launch_shared<CQ_DTYPE_Q5K>(ma, (unsigned)tiles, a, m, s);
    default: return launch_shared<CQ_DTYPE_Q6K>(ma, (unsigned)tiles, a, m, s);
    }
}
