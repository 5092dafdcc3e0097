// Prefill GEMM for the 32-element-block types (Q8_0 and Q4_0 weights, Q8_0 activations) on the int8
// MFMA: y[m, n] = x[m, k] . W[n, k]^T with the arithmetic of the reference's CPU matmul
// (k_quants.rs:1842-1883 with vec_dot :237-254 for Q4_0, :631-649 for Q8_0): per block the integer
// sum of 32 products, times the two block scales.  Replaces the reference's MMQ kernels for these
// types (candle-kernels/src/quantized.cu:436-544, launched from quantized/cuda.rs:298-365).
//
// A 32-element block is exactly one K-slice of v_mfma_i32_32x32x32_i8, so the integer of every
// (activation row, weight row, block) is one MFMA result element, I (Q4_0 nibbles go in as q - 8, so
// no correction term is left).  Its scale d8[row, block] * dw[col, block] is an outer product: a
// second MFMA lays it out in the accumulator layout (v_mfma_f32_32x32x8_f16 with one non-zero K-slot: both scales are f16
// values, and their product, subnormal factors included, is exact in f32), and the VALU
// work per element is one conversion and one fma.
// Bound by vector issue.  ns a step of the two waves of a SIMD (a tile and block of each) in a loop of nothing but steps, the scales as two bf16
// pieces each (v_mfma_f32_32x32x16_bf16: three instructions for the operand, three for the zeros beside it) -> as f16: Q8_0 70.9 -> 62.8, Q4_0
// 68.5 -> 61.0; without the second MFMA 55.6.  Whole calls, weights from HBM, us: Q8_0 11008 x 4096 at 4096 / 512 / 64 rows 520 -> 483, 99.3 -> 93.7,
// 27.7 -> 27.6, Q4_0 4096 x 4096 at 512 / 1024 rows 37.2 -> 35.5, 61.3 -> 57.4, 11008 x 4096 at 4096 499 -> 459, Q5_0 4096 x 11008 at 700
// 154.6 -> 144.8.  (The next step's weight operands read under this step's last tile instead of behind the barrier: level to 2 % slower.)
//
// Work split as in the K-quant tile kernel (gemm.hip): a workgroup of eight waves covers 32*MT
// activation rows x 256 weight rows, a wave owns 32 weight rows; per 256-element step of K the
// activations (shared) and the wave's weight bytes go from global memory straight into LDS
// (buffer_load ... lds, 8 rows x 128 B per instruction, 16-byte chunks XOR-swizzled by the row),
// activations double buffered one step ahead.  Where that gives few workgroups K is split inside them (gemm32_kh_kernel, and
// for up to 32 rows gemm32_few_kernel) or over blockIdx.z, the partial results then added atomically into a zeroed output.
#include "qhip_internal.h"
#include <type_traits>

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef void __attribute__((address_space(3))) *lptr_t;
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));   // (rows of whole 64-element pairs of blocks)

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t wave_rsrc(const void *base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, -1, 0x00020000);
}
// lane l reads 16 (4) bytes at base + off, they land at lds + 16*l (4*l; base and lds wave-uniform)
__device__ __forceinline__ void dma16(const void *base, uint32_t off, uint8_t *lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(wave_rsrc(base), (lptr_t)lds, 16, (int)off, 0, 0, 0);
}
__device__ __forceinline__ void dma4(const void *base, uint32_t off, uint8_t *lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(wave_rsrc(base), (lptr_t)lds, 4, (int)off, 0, 0, 0);
}
// the same marked non-temporal: bytes that the launch reads once
__device__ __forceinline__ void dma16_once(const void *base, uint32_t off, uint8_t *lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(wave_rsrc(base), (lptr_t)lds, 16, (int)off, 0, 0, 2);
}

// LDS: two activation stages, then one weight buffer per wave.
//   act : [MT tiles][2 K-halves][4 row groups][8 rows][8 chunks of 16 B]   chunk c of row r sits at c ^ (r%8) ^ ((r/8)%2)
//         (a 16-byte read serves sixteen lanes at a time, rows of two groups: with c ^ (r%8) alone they meet in half the banks,
//         8.3 cycles a read instead of 5.0)
//   d8  : [MT tiles][8 blocks][32 rows] f32, out of the block-major plane (a lane per row reads one word of consecutive ones)
//   wgt : per wave, Q8_0: [2 K-halves][4 row groups][8 rows][8 chunks]; Q4_0: [4 row groups][8 rows][8 chunks]
template <int DT, int MT> struct Tile {
    static constexpr int kAct = MT * 8 * 1024;
    static constexpr int kD8 = MT * 32 * 32;
    static constexpr int oD8 = kAct;
    static constexpr int kStage = kAct + kD8;
    static constexpr int kWgtWave = DT == CQ_DTYPE_Q8_0 ? 8192 : 4096;
    static constexpr int oWgt = 2 * kStage;
    static constexpr int kTotal = oWgt + kWaves * kWgtWave;
};

// What the sums are multiplied by on their way out: a power of two, exact (the scales are f16 values: no sum comes near the range of f32).
template <int DT> constexpr float kUnit = DT == CQ_DTYPE_Q4_0 ? 0.0625f : 1.0f;

struct LaneGeo {
    uint32_t row_off;    // copy of 8 rows x 128 B with a row pitch of k bytes: (l/8)*k + ((l%8) ^ (l/8))*16; odd row groups: ^ 16
    uint32_t w4_off;     // the same with the Q4_0 row pitch of k/2 bytes
    uint32_t d8_off;     // copy of 8 blocks x 32 rows of scales: block l/8, rows 4*(l%8)..; ANYROW two blocks: block l/32, row l%32
    uint32_t col[4];     // operand read: byte offset of chunk 2j+h of row l%32 inside a [4][8][8] x 16 B image
    uint32_t col4[8];    // Q4_0: chunk s of row l%32 (the 16 bytes of block s)
};

template <bool ANYROW> __device__ __forceinline__ LaneGeo lane_geo(int lane, int64_t k, int64_t m_stride) {
    LaneGeo g;
    const uint32_t r8 = lane >> 3, c8 = lane & 7;
    g.row_off = r8 * (uint32_t)k + ((c8 ^ r8) << 4);
    g.w4_off = r8 * (uint32_t)(k >> 1) + ((c8 ^ r8) << 4);
    g.d8_off = ANYROW ? ((uint32_t)(lane >> 5) * (uint32_t)m_stride + (uint32_t)(lane & 31)) * 4u
                      : ((uint32_t)(lane >> 3) * (uint32_t)m_stride + (uint32_t)(lane & 7) * 4u) * 4u;
    const uint32_t r = lane & 31, h = lane >> 5;
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) g.col[j] = (r >> 3) * 1024u + (r & 7) * 128u + (((2 * j + h) ^ (r & 7) ^ ((r >> 3) & 1)) << 4);
#pragma unroll
    for (uint32_t s = 0; s < 8; s++) g.col4[s] = (r >> 3) * 1024u + (r & 7) * 128u + ((s ^ (r & 7) ^ ((r >> 3) & 1)) << 4);
    return g;
}

// This wave's share of the activation copies of K step b into stage `buf`.  ANYROW: tiles begin at any row (a grouped launch),
// where the scales of a block lie on four bytes and are copied word by word; otherwise rows and plane pitch are whole
// 32-row groups, and 16 bytes a lane take a tile's scales in one copy.
template <int DT, int MT, bool ANYROW>
__device__ __forceinline__ void stage_acts(uint8_t *buf, const cq_act_view &a, const LaneGeo &g, int64_t k, int64_t m0,
                                           int64_t b, int wave) {
    typedef Tile<DT, MT> T;
#pragma unroll
    for (int j = 0; j < MT * 8 / kWaves; j++) {
        const int idx = wave + kWaves * j;           // = (t*2 + kh)*4 + rg
        const int rg = idx & 3, kh = (idx >> 2) & 1, t = idx >> 3;
        dma16(a.qs + (m0 + t * 32 + rg * 8) * k + b * 256 + kh * 128, g.row_off ^ (uint32_t)((rg & 1) << 4), buf + idx * 1024);
    }
#pragma unroll
    for (int t = 0; t < MT; t++) {
        if (t + 4 != wave) continue;
        const float *d8 = a.dT + b * 8 * a.m_stride + m0 + t * 32;
        if (ANYROW) {
#pragma unroll
            for (int i = 0; i < 4; i++) dma4(d8 + 2 * i * a.m_stride, g.d8_off, buf + T::oD8 + t * 1024 + i * 256);
        } else {
            dma16(d8, g.d8_off, buf + T::oD8 + t * 1024);
        }
    }
}

// This wave's 32 weight rows of K step b into its own buffer.
template <int DT, bool ONCE>
__device__ __forceinline__ void stage_weights(uint8_t *wl, const cq_weight &w, const LaneGeo &g, int64_t n_tile, int64_t b) {
    const int64_t k = w.k;
    if (DT == CQ_DTYPE_Q8_0) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int rg = i & 3, kh = i >> 2;
            if (ONCE) dma16_once(w.p0 + (n_tile + rg * 8) * k + b * 256 + kh * 128, g.row_off ^ (uint32_t)((rg & 1) << 4), wl + i * 1024);
            else dma16(w.p0 + (n_tile + rg * 8) * k + b * 256 + kh * 128, g.row_off ^ (uint32_t)((rg & 1) << 4), wl + i * 1024);
        }
    } else {
#pragma unroll
        for (int rg = 0; rg < 4; rg++) {
            if (ONCE) dma16_once(w.p0 + (n_tile + rg * 8) * (k >> 1) + b * 128, g.w4_off ^ (uint32_t)((rg & 1) << 4), wl + rg * 1024);
            else dma16(w.p0 + (n_tile + rg * 8) * (k >> 1) + b * 128, g.w4_off ^ (uint32_t)((rg & 1) << 4), wl + rg * 1024);
        }
    }
}

// Weight operands of the eight blocks of a K step out of the wave's buffer (which is then free for the next step).
template <int DT> __device__ __forceinline__ void step_weights(const uint8_t *wl, const LaneGeo &g, int h, v4i (&bw)[8]) {
    if (DT == CQ_DTYPE_Q8_0) {
#pragma unroll
        for (int s = 0; s < 8; s++) bw[s] = *(const v4i *)(wl + (s >> 2) * 4096 + g.col[s & 3]);
    } else {
#pragma unroll
        for (int s = 0; s < 8; s++) {
            // block s: 16 bytes, low nibbles = elements 0..15 (h = 0), high nibbles = elements 16..31; as 16 * (q - 8), the
            // nibble in the upper half of its byte: two instructions a word (kUnit takes the 1/16 out of the results)
            const v4i q = *(const v4i *)(wl + g.col4[s]);
#pragma unroll
            for (int i = 0; i < 4; i++) bw[s][i] = (int)((((uint32_t)q[i] << (4 - 4 * h)) & 0xF0F0F0F0u) ^ 0x80808080u);
        }
    }
}

// One K step: the eight blocks of `bw` against the MT tiles of the stage `cur`.  `dcur`: the lane's weight row's eight f16 block
// scales; nv: blocks of the step that exist (SHORT).
// LOWER: at most sixteen rows of the last tile are live, and its upper sixteen (results 8..15) are not scaled.
template <int DT, int MT, bool DUMP, bool SHORT, bool LOWER = false>
__device__ __forceinline__ void step_mac(const uint8_t *cur, const LaneGeo &g, const v4i (&bw)[8], const u32x4_a4 dcur, int nv, int h, int col,
                                         v16f (&out)[MT], const cq_weight &w, int64_t m0, int64_t m, int64_t n, int64_t b, cq_mfma_dump dump) {
    typedef Tile<DT, MT> T;
    // scale operand of block s: the f16 scale in the one K-slot that is not zero (lanes 0..31)
    // A last step of fewer than eight blocks: what follows the rows in memory (other rows, other planes) was copied
    // with them, and both scales of the blocks that do not exist are zero.
    const uint32_t dwords[4] = {dcur.x, dcur.y, dcur.z, dcur.w};
    v4h dw[8];
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const uint32_t bits = s & 1 ? dwords[s >> 1] >> 16 : dwords[s >> 1] & 0xffffu;
        const v2u pk = {h == 0 && (!SHORT || s < nv) ? bits : 0u, 0u};
        dw[s] = __builtin_bit_cast(v4h, pk);
    }

    // steps q = (tile t, block s): the two MFMAs of step q, and in their shadow the scaling of step q-1
    auto afrag = [&](int q) -> v4i {
        const int t = q >> 3, s = q & 7;
        return *(const v4i *)(cur + g.col[s & 3] + (t * 2 + (s >> 2)) * 4096);
    };
    // activation scale of (row l%32 of tile t, block s): read two steps ahead, and only turned into
    // the MFMA operand in the step that uses it, so that no step
    // waits for the read it has just issued
    auto d8raw = [&](int q) -> float {
        const int t = q >> 3, s = q & 7;
        const float v = *(const float *)(cur + T::oD8 + t * 1024 + s * 128 + col * 4);
        return !SHORT || s < nv ? v : 0.0f;
    };
    auto d8frag = [&](float v) -> v4h {
        // an f16 value, in the K-slot that the weight's scale is in; in slots where that has zeros stays what the register holds (finite where the
        // scale is)
        const _Float16 d = (_Float16)v;
        const v2u pk = {(uint32_t)__builtin_bit_cast(uint16_t, d), __float_as_uint(v)};
        return __builtin_bit_cast(v4h, pk);
    };
    v16i acc[2];
    v16f sc[2];
    v4i av[3];
    float dv[3];
    av[0] = afrag(0); av[1] = afrag(1);
    dv[0] = d8raw(0); dv[1] = d8raw(1);
    const v16i zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const v16f zerof = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q <= MT * 8; q++) {
        if (q + 2 < MT * 8) { av[(q + 2) % 3] = afrag(q + 2); dv[(q + 2) % 3] = d8raw(q + 2); }
        if (q < MT * 8) {
            acc[q & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[q % 3], bw[q & 7], zero, 0, 0, 0);
            sc[q & 1] = __builtin_amdgcn_mfma_f32_32x32x8f16(d8frag(dv[q % 3]), dw[q & 7], zerof, 0, 0, 0);
        }
        // keeps the MFMAs in front of the scaling below: left alone, the scheduler sinks them to the end
        // of the step, and the next step then starts by waiting for their results
        __builtin_amdgcn_sched_barrier(0);
        if (q > 0) {
            const int p = (q - 1) & 1, t = (q - 1) >> 3;
#pragma unroll
            for (int i = 0; i < (LOWER && t == MT - 1 ? 8 : 16); i++) {
                if (DUMP) {   // (whole K steps only)
                    const int64_t row = m0 + t * 32 + (i >> 2) * 8 + h * 4 + (i & 3);
                    if (row < m) dump.i[(row * w.n + n) * (w.k >> 5) + b * 8 + ((q - 1) & 7)] = DT == CQ_DTYPE_Q4_0 ? acc[p][i] >> 4 : acc[p][i];
                } else {
                    out[t][i] = __builtin_fmaf((float)acc[p][i], sc[p][i], out[t][i]);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// DUMP (verification): the block integers are stored through `dump` instead of the result through `y`.
// ONCE: a launch with a single row tile (up to 32 rows), which reads every weight byte once.
// SHORT: K is no multiple of 256, the last step has fewer than eight blocks.
template <int DT, int MT, bool DUMP, bool ONCE, bool SHORT, bool ANYROW = false>
__device__ __forceinline__ void gemm32_body(const cq_weight &w, const cq_act_view &a, int64_t bx, int64_t m0, int64_t m, float *__restrict__ y,
                                            int ksplit, bool stream, cq_mfma_dump dump) {
    typedef Tile<DT, MT> T;
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h = lane >> 5, col = lane & 31;
    const int64_t k = w.k, ks = (k + 255) >> 8;         // K steps of 256 elements; the last one may be shorter
    const int64_t n_own = (bx * kWaves + wave) * 32;
    const bool n_ok = n_own < w.n;                      // wave-uniform; a wave past the last row only helps with the copies
    // fewer than 32 rows left: the tile begins earlier, at row n - 32, and only the wave's own share is stored
    const int64_t n_tile = n_own + 32 <= w.n ? n_own : w.n - 32;
    const int64_t n = n_tile + col;
    const int64_t nc = n_ok ? n : 0;
    const int64_t b0 = ks * blockIdx.z / ksplit, b1 = ks * (blockIdx.z + 1) / ksplit;
    const LaneGeo g = lane_geo<ANYROW>(lane, k, a.m_stride);
    uint8_t *__restrict__ wl = smem + T::oWgt + wave * T::kWgtWave;
    const uint16_t *dplane = (const uint16_t *)w.p1;    // f16 block scales [n][k/32]

    v16f out[MT];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int i = 0; i < 16; i++) out[t][i] = 0.0f;

    stage_acts<DT, MT, ANYROW>(smem, a, g, k, m0, b0, wave);
    if (n_ok) stage_weights<DT, ONCE>(wl, w, g, n_tile, b0);
    u32x4_a4 dnext = *(const u32x4_a4 *)(dplane + nc * (k >> 5) + b0 * 8);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();

    for (int64_t b = b0; b < b1; b++) {
        const uint8_t *__restrict__ cur = smem + ((b - b0) & 1) * T::kStage;
        uint8_t *__restrict__ nxt = smem + (((b - b0) & 1) ^ 1) * T::kStage;
        const bool more = b + 1 < b1;
        if (more) stage_acts<DT, MT, ANYROW>(nxt, a, g, k, m0, b + 1, wave);
        if (n_ok) {
            v4i bw[8];
            step_weights<DT>(wl, g, h, bw);
            const u32x4_a4 dcur = dnext;
            if (more) {
                stage_weights<DT, ONCE>(wl, w, g, n_tile, b + 1);
                dnext = *(const u32x4_a4 *)(dplane + nc * (k >> 5) + (b + 1) * 8);
            }
            step_mac<DT, MT, DUMP, SHORT>(cur, g, bw, dcur, (int)((k >> 5) - b * 8), h, col, out, w, m0, m, n, b, dump);
        }
        __builtin_amdgcn_s_waitcnt(0);   // the next stage and the wave's next weights have landed in LDS
        __syncthreads();
    }

    if (n_ok && !DUMP) {
        cq_put_results(ksplit, stream, [&](auto how) {
#pragma unroll
            for (int t = 0; t < MT; t++) {
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int64_t row = m0 + t * 32 + (i >> 2) * 8 + h * 4 + (i & 3);
                    if (row < m && n >= n_own) cq_put_result<decltype(how)::value>(&y[row * w.n + n], out[t][i] * kUnit<DT>);
                }
            }
        });
    }
}

template <int DT, int MT, bool DUMP, bool ONCE, bool SHORT>
__global__ void __launch_bounds__(kThreads) gemm32_kernel(cq_weight w, cq_act_view a, int64_t m, float *__restrict__ y, int ksplit,
                                                          int strips, int stream, cq_mfma_dump dump) {
    const cq_tile t = cq_tile_at(blockIdx.x, blockIdx.y, gridDim.x, gridDim.y, strips);
    gemm32_body<DT, MT, DUMP, ONCE, SHORT>(w, a, t.x, (int64_t)t.y * (MT * 32), m, y, ksplit, stream != 0, dump);
}

// Few column tiles: K halved inside the workgroup (as gemm_kh_kernel of gemm.hip).  A workgroup covers 128 weight rows x 32*MT
// activation rows; waves 0..3 take the first half of the K steps, waves 4..7 the second half for the same weight rows, and
// the partial tiles meet in LDS, first half + second half: twice the workgroups at the same tile height, no atomic additions.
// Bound, as above, by vector issue (one conversion and one fma per element and block, two thirds of the instructions).  Whole calls, us, before
// -> here: Q4_0 32003 x 3200 at 77 rows (251 workgroups of 96 rows for 252 of 64, the upper ones nearly empty) 54.8 -> 42.1,
// 29731 x 4864 at 90 rows 69.6 -> 51.9; with the scaling of sixteen rows of padding left out (LOWER) 42.2 -> 40.5 at 77 rows, 29731 x 4864
// 50.7 -> 48.7; Q8_0 4096 x 4096 at 512 rows 40.7 -> 36.1, 8192 x 2048 at 60 rows 16.1 -> 14.4.
template <int DT, int MT> struct TileKH {
    typedef Tile<DT, MT> T;
    static constexpr int oWgt = 4 * T::kStage;   // two stages of one part per half
    static constexpr int kTotal = oWgt + kWaves * T::kWgtWave;
    static_assert(kTotal <= 160 * 1024 && MT * 4096 * (kWaves / 2) <= oWgt, "the stages fit the LDS, the partial tiles the stages");
};
// Row tiles that gemm32_kh_kernel's stages leave room for beside the weights (Q8_0: 8 KiB a wave).
template <int DT> constexpr int kh_tallest() { return DT == CQ_DTYPE_Q4_0 ? 3 : 2; }
template <int DT, int MT, bool DUMP, bool SHORT, bool LOWER>
__global__ void __launch_bounds__(kThreads) gemm32_kh_kernel(cq_weight w, cq_act_view a, int64_t m, float *__restrict__ y, int stream,
                                                             cq_mfma_dump dump) {
    typedef Tile<DT, MT> T;
    typedef TileKH<DT, MT> TK;
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int colw = wave & 3, half = wave >> 2, h = lane >> 5, col = lane & 31;
    const int64_t k = w.k, m0 = (int64_t)blockIdx.y * (MT * 32);
    const int ks = (int)((k + 255) >> 8), nh = (ks + 1) / 2;
    const int64_t n_own = ((int64_t)blockIdx.x * (kWaves / 2) + colw) * 32;
    const bool n_ok = n_own < w.n;
    const int64_t n_tile = n_own + 32 <= w.n ? n_own : w.n - 32, n = n_tile + col;
    const int first = half ? nh : 0, count = half ? ks - nh : nh;
    const LaneGeo g = lane_geo<false>(lane, k, a.m_stride);
    uint8_t *__restrict__ wl = smem + TK::oWgt + wave * T::kWgtWave;
    const uint16_t *dplane = (const uint16_t *)w.p1 + (n_ok ? n : 0) * (k >> 5);

    v16f out[MT];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int i = 0; i < 16; i++) out[t][i] = 0.0f;

    stage_acts<DT, MT, false>(smem, a, g, k, m0, 0, wave);
    if (ks > nh) stage_acts<DT, MT, false>(smem + T::kStage, a, g, k, m0, nh, wave);
    u32x4_a4 dnext = {};
    if (n_ok && count > 0) {
        stage_weights<DT, false>(wl, w, g, n_tile, first);
        dnext = *(const u32x4_a4 *)(dplane + first * 8);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    for (int it = 0; it < nh; it++) {
        const uint8_t *__restrict__ cur = smem + (2 * (it & 1) + half) * T::kStage;
        uint8_t *__restrict__ nxt = smem + 2 * ((it & 1) ^ 1) * T::kStage;
        if (it + 1 < nh) stage_acts<DT, MT, false>(nxt, a, g, k, m0, it + 1, wave);
        if (nh + it + 1 < ks) stage_acts<DT, MT, false>(nxt + T::kStage, a, g, k, m0, nh + it + 1, wave);
        if (n_ok && it < count) {
            const int b = first + it;
            v4i bw[8];
            step_weights<DT>(wl, g, h, bw);
            const u32x4_a4 dcur = dnext;
            if (it + 1 < count) {
                stage_weights<DT, false>(wl, w, g, n_tile, b + 1);
                dnext = *(const u32x4_a4 *)(dplane + (b + 1) * 8);
            }
            step_mac<DT, MT, DUMP, SHORT, LOWER>(cur, g, bw, dcur, (int)(k >> 5) - b * 8, h, col, out, w, m0, m, n, b, dump);
        }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
    }
    if (DUMP) return;
    // (the stages are free: every wave is past its last read)
    float *part = (float *)smem + (size_t)colw * (MT * 16 * 64);
    if (half == 1) {
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int i = 0; i < 16; i++) part[(t * 16 + i) * 64 + lane] = out[t][i];
    }
    __syncthreads();
    if (half == 0 && n_ok) {
        cq_put_results(1, stream != 0, [&](auto how) {
#pragma unroll
            for (int t = 0; t < MT; t++) {
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int64_t row = m0 + t * 32 + (i >> 2) * 8 + h * 4 + (i & 3);
                    if (row < m && n >= n_own) cq_put_result<decltype(how)::value>(&y[row * w.n + n], (out[t][i] + part[(t * 16 + i) * 64 + lane]) * kUnit<DT>);
                }
            }
        });
    }
}

// Up to 32 activation rows: every wave by itself.  A workgroup covers 32*CW weight rows, its waves share the K steps: wave p * CW + c
// takes steps p, p + KS, ... (KS = 8 / CW) of column tile c into a buffer of its own, activations included, so that no wave
// waits for another before the end, where the KS partial tiles of each column tile are added in order.  No atomic additions, and
// nothing for the quantizer to clear.  Bound by the weights' way in: a step's weights are requested while the one before is
// contracted, its activations behind it (there is no LDS for two sets).  Whole calls, us, K split over workgroups -> here: Q4_0 14336 x 4096 at
// 21 rows 18.2 -> 14.8, Q8_0 20.9 -> 19.5; more partial tiles than that cost more than they give (Q8_0 8192 x 8192 as 256
// workgroups of one column tile 19.8 -> 24.0).
template <int DT> struct Few {
    typedef Tile<DT, 1> T;
    static constexpr int kWave = T::kStage + T::kWgtWave;
    static constexpr int kTotal = kWaves * kWave;
};
template <int DT, int CW, bool DUMP, bool ONCE, bool SHORT>
__global__ void __launch_bounds__(kThreads) gemm32_few_kernel(cq_weight w, cq_act_view a, int64_t m, float *__restrict__ y, cq_mfma_dump dump) {
    typedef Tile<DT, 1> T;
    constexpr int KS = kWaves / CW;
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int colw = wave % CW, part = wave / CW, h = lane >> 5, col = lane & 31;
    const int64_t k = w.k;
    const int ks = (int)((k + 255) >> 8), groups = (int)((m + 7) / 8);
    const int64_t n_own = ((int64_t)blockIdx.x * CW + colw) * 32;
    const bool n_ok = n_own < w.n;
    const int64_t n_tile = n_own + 32 <= w.n ? n_own : w.n - 32, n = n_tile + col;
    const LaneGeo g = lane_geo<false>(lane, k, a.m_stride);
    uint8_t *__restrict__ act = smem + wave * Few<DT>::kWave;
    uint8_t *__restrict__ wl = act + T::kStage;
    const uint16_t *dplane = (const uint16_t *)w.p1 + (n_ok ? n : 0) * (k >> 5);

    v16f out[1];
#pragma unroll
    for (int i = 0; i < 16; i++) out[0][i] = 0.0f;
    auto copy_acts = [&](int b) {
#pragma unroll
        for (int idx = 0; idx < 8; idx++) {
            const int rg = idx & 3, kh = idx >> 2;
            if (rg < groups) dma16(a.qs + (int64_t)(rg * 8) * k + b * 256 + kh * 128, g.row_off ^ (uint32_t)((rg & 1) << 4), act + idx * 1024);
        }
        dma16(a.dT + (int64_t)b * 8 * a.m_stride, g.d8_off, act + T::oD8);
    };
    if (n_ok && part < ks) {
        u32x4_a4 dnext = *(const u32x4_a4 *)(dplane + part * 8);
        stage_weights<DT, ONCE>(wl, w, g, n_tile, part);
        copy_acts(part);
#pragma nounroll
        for (int b = part; b < ks; b += KS) {
            __builtin_amdgcn_s_waitcnt(0);   // the step's copies have landed
            const uint8_t *__restrict__ cur = act;
            v4i bw[8];
            step_weights<DT>(wl, g, h, bw);
            const u32x4_a4 dcur = dnext;
            if (b + KS < ks) {
                __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the reads above are done with the buffer
                dnext = *(const u32x4_a4 *)(dplane + (b + KS) * 8);
                stage_weights<DT, ONCE>(wl, w, g, n_tile, b + KS);
            }
            step_mac<DT, 1, DUMP, SHORT>(cur, g, bw, dcur, (int)(k >> 5) - b * 8, h, col, out, w, 0, m, n, b, dump);
#pragma unroll
            for (int i = 0; i < 16; i++) asm volatile("" : "+v"(out[0][i]));   // (keeps the arithmetic in front of the branch: it would sink behind it, with all it holds)
            if (b + KS < ks) {
                __builtin_amdgcn_s_waitcnt(0xC07F);
                copy_acts(b + KS);
            }
        }
    }
    if (DUMP) return;
    if constexpr (KS > 1) {
        float *mine = (float *)act;
#pragma unroll
        for (int i = 0; i < 16; i++) mine[i * 64 + lane] = out[0][i];
        __syncthreads();
    }
    // wave p * CW + c adds and stores registers 16 / KS * p .. of column tile c
    if (!n_ok || n < n_own) return;
#pragma unroll
    for (int j = 0; j < 16 / KS; j++) {
        const int i = part * (16 / KS) + j;
        float v = KS > 1 ? 0.0f : out[0][j];
        if constexpr (KS > 1) {
#pragma unroll
            for (int p = 0; p < KS; p++) v += *(const float *)(smem + (p * CW + colw) * Few<DT>::kWave + (i * 64 + lane) * 4);
        }
        const int64_t row = (i >> 2) * 8 + h * 4 + (i & 3);
        if (row < m) y[row * w.n + n] = v * kUnit<DT>;
    }
}

// 128-row tiles in whole rounds of workgroups, what is left of them in tiles of 32 * TAIL rows (as gemm_tail_kernel of
// gemm.hip): `whole` of the gx x row tiles, in strips, are taken whole, the others by 4 / TAIL workgroups each.
template <int DT, int TAIL, bool DUMP, bool SHORT>
__global__ void __launch_bounds__(kThreads) gemm32_tail_kernel(cq_weight w, cq_act_view a, int64_t m, float *__restrict__ y, uint32_t gx,
                                                               uint32_t whole, int stream, cq_mfma_dump dump) {
    const uint32_t id = blockIdx.x, gy = (uint32_t)((m + 127) / 128);
    if (id < whole) {
        const cq_tile t = cq_tile_in_strips(cq_tile_of_xcd(id, whole), gx, gy);
        gemm32_body<DT, 4, DUMP, false, SHORT>(w, a, t.x, (int64_t)t.y * 128, m, y, 1, stream != 0, dump);
    } else {
        const uint32_t at = cq_tile_of_xcd(id - whole, gridDim.x - whole);
        const cq_tile t = cq_tile_in_strips(whole + at / (4 / TAIL), gx, gy);
        const int64_t m0 = (int64_t)t.y * 128 + at % (4 / TAIL) * (32 * TAIL);
        if (m0 < m) gemm32_body<DT, TAIL, DUMP, false, SHORT>(w, a, t.x, m0, m, y, 1, stream != 0, dump);
    }
}

// Mixture-of-experts form: blockIdx.y walks a table of tiles of 32*MT rows of the expert-sorted activation rows; each tile names
// its expert's weights (as gemm_grouped_kernel of gemm.hip).
template <int DT, int MT, bool SHORT>
__global__ void __launch_bounds__(kThreads) gemm32_grouped_kernel(cq_group_args ga, cq_act_view a, float *__restrict__ y, int ksplit) {
    const int tile = blockIdx.y;
    const cq_weight w = ga.w[ga.expert[tile]];
    gemm32_body<DT, MT, false, MT == 1, SHORT, true>(w, a, blockIdx.x, ga.row0[tile], min(ga.row0[tile] + 32 * MT, ga.row_end[tile]), y, ksplit, false,
                                               cq_mfma_dump{nullptr, nullptr, 0});
}

// Tile height (MT x 32 activation rows per workgroup) and K split of a launch, from a cost model fitted to
// measurements (Q8_0, 256 CUs; unit 1/16 us): a workgroup spends 10 units per 256-element K step on its
// weights and 23 per 32-row tile on it, 24 on starting and finishing; workgroups run one per CU, in rounds;
// a split launch adds every part to the output atomically, which moves about 1.1 TB/s.
// The launches that split K inside the workgroup are priced beside them (half the steps at 11 + 22 units a row tile, 40 for start,
// end and meeting; up to 32 rows 30 units a step of a wave and 29), taken where one round of workgroups does it and the sum is at least 5 %
// lower.  Against a sweep of both on 1857 cases (512..32000 weight rows, K 512..14336, 17..2048 rows) the choice is 0.5 % off the
// better one on average (the tile launches alone 8 %), 5.5 % faster than they are and 7 % slower at worst (Q8_0 512 x 1024 at 512 rows, 0.8 us).
struct Plan {
    int mt, ksplit;
    int tail = 0;   // 1, 2: gemm32_tail_kernel, the last round's tiles in heights of 32 * tail rows
    int kh = 0;     // 1: gemm32_kh_kernel
    int few = 0;    // 1, 2, 4, 8: gemm32_few_kernel with that many column tiles a workgroup
    double work = 0.0, merge = 0.0;   // the cost: workgroups, adding up the parts
};
Plan pick_plan(const cq_weight *w, int64_t m) {
    const int64_t gx = (w->n + kWaves * 32 - 1) / (kWaves * 32), ks_total = (w->k + 255) >> 8, cus = cq_num_cus();
    const double atomic_pass = (double)m * (double)w->n * 4.0 / 1.1e6 * 16.0;   // bytes / (1.1e6 bytes per us) in units
    Plan best{1, 1};
    double best_cost = 0.0;
    bool first = true;
    for (int mt = 4; mt >= 1; mt >>= 1) {
        if (mt > 1 && m <= 16 * mt) continue;   // half the height holds all rows
        const int64_t tiles = gx * ((m + mt * 32 - 1) / (mt * 32));
        for (int ks = 1; ks <= 16; ks *= 2) {
            if (ks > 1 && ks_total / ks < 2) break;
            if (ks > 1 && cq_no_split_k()) break;   // CQ_FLAG_DETERMINISTIC
            const int64_t rounds = (tiles * ks + cus - 1) / cus;
            const double merge = ks > 1 ? ks * atomic_pass : 0.0;
            double cost = (double)rounds * ((double)((ks_total + ks - 1) / ks) * (10.0 + 23.0 * mt) + 24.0) + merge;
            // A last round that is at most half full (or a quarter), in shorter tiles.  Whole calls, us, one height -> two: Q8_0
            // 11008 x 4096 at 4096 / 1024 rows 610 -> 580 / 181 -> 163, 5120 x 5120 at 2000 229 -> 178, 8448 x 2048 at 1024
            // 99 -> 77; Q4_0 4096 x 14336 at 2300 512 -> 456.
            int tail = 0;
            const int64_t left = tiles % cus;
            for (int t = 2; t >= 1 && mt == 4 && ks == 1 && rounds > 1 && left > 0 && left * (4 / t) <= cus; t--) {
                cost = (double)(rounds - 1) * ((double)ks_total * (10.0 + 23.0 * 4) + 24.0) + ((double)ks_total * (10.0 + 23.0 * t) + 24.0);
                tail = t;
            }
            if (first || cost < best_cost) {
                best = Plan{mt, ks, tail, 0, 0, cost - merge, merge};
                best_cost = cost;
                first = false;
            }
        }
    }
    const double limit = 0.95 * best_cost;
    best_cost = limit;
    for (int mt = w->dtype == CQ_DTYPE_Q4_0 ? kh_tallest<CQ_DTYPE_Q4_0>() : kh_tallest<CQ_DTYPE_Q8_0>(); mt >= 1; mt--) {
        if (mt > 1 && m <= 32 * (mt - 1)) continue;   // a row tile less holds all rows
        if (mt == 3 && (m + 95) / 96 * 96 > (m + 127) / 128 * 128) continue;   // (the workspace's rows are padded to 128)
        if ((w->n + 127) / 128 * ((m + mt * 32 - 1) / (mt * 32)) > cus) continue;
        const double cost = (double)((ks_total + 1) / 2) * (11.0 + 22.0 * mt) + 40.0;
        if (cost < best_cost) {
            best = Plan{mt, 1, 0, 1, 0, cost, 0.0};
            best_cost = cost;
        }
    }
    for (int cw = 8; cw >= 1 && m <= 32; cw >>= 1) {
        const int64_t groups = (w->n + 32 * cw - 1) / (32 * cw), parts = kWaves / cw;
        if (groups > (cw == 1 && w->dtype == CQ_DTYPE_Q8_0 ? cus / 2 : cus)) continue;
        const double cost = (double)((ks_total + parts - 1) / parts) * 30.0 + 29.0;
        if (cost < best_cost) {
            best = Plan{1, 1, 0, 0, cw, cost, 0.0};
            best_cost = cost;
        }
    }
    return best;
}

// DUMP (here and below): the same launch (kernel, tile height, K split; copies never marked non-temporal) storing the block integers through
// `d`; y is not touched.
template <int DT, int MT, bool DUMP, bool ONCE, bool SHORT>
hipError_t launch_inst(const cq_weight *w, cq_act_view a, int64_t m, float *y, int ksplit, cq_mfma_dump d, hipStream_t s) {
    const size_t lds = Tile<DT, MT>::kTotal;
    if (hipError_t e = cq_ensure_lds<gemm32_kernel<DT, MT, DUMP, ONCE, SHORT>>(w->dev, lds); e != hipSuccess) return e;
    const dim3 grid((unsigned)((w->n + kWaves * 32 - 1) / (kWaves * 32)), (unsigned)((m + MT * 32 - 1) / (MT * 32)), (unsigned)ksplit);
    CQ_LAUNCH((gemm32_kernel<DT, MT, DUMP, ONCE, SHORT>), grid, kThreads, lds, s, *w, a, m, y, ksplit, cq_tiles_in_strips((int64_t)grid.x * grid.y, ksplit),
              (int)cq_streams_result(w, m), d);
    return hipGetLastError();
}
template <int DT, int TAIL, bool DUMP, bool SHORT>
hipError_t launch_tail(const cq_weight *w, cq_act_view a, int64_t m, float *y, cq_mfma_dump d, hipStream_t s) {
    const size_t lds = Tile<DT, 4>::kTotal;
    if (hipError_t e = cq_ensure_lds<gemm32_tail_kernel<DT, TAIL, DUMP, SHORT>>(w->dev, lds); e != hipSuccess) return e;
    const int64_t gx = (w->n + kWaves * 32 - 1) / (kWaves * 32), tiles = gx * ((m + 127) / 128), whole = tiles / cq_num_cus() * cq_num_cus();
    CQ_LAUNCH((gemm32_tail_kernel<DT, TAIL, DUMP, SHORT>), (unsigned)(whole + (tiles - whole) * (4 / TAIL)), kThreads, lds, s, *w, a, m, y,
              (uint32_t)gx, (uint32_t)whole, (int)cq_streams_result(w, m), d);
    return hipGetLastError();
}
// A single row tile over that many bytes of weights and more: the copies marked non-temporal (measured at 17 and 32 rows:
// 3-7 % faster from there on, 3-5 % slower below).
constexpr int64_t kOnceBytes = 40000000;
template <int DT, int MT, bool DUMP>
hipError_t launch_mt(const cq_weight *w, cq_act_view a, int64_t m, float *y, int ksplit, bool y_cleared, cq_mfma_dump d,
                     hipStream_t s) {
    if constexpr (DUMP) {
        return launch_inst<DT, MT, true, false, false>(w, a, m, y, ksplit, d, s);   // (whole K steps only)
    } else {
        if (ksplit > 1 && !y_cleared) {
            hipError_t e = cq_launch_fill_zero(y, m * w->n, s);
            if (e != hipSuccess) return e;
        }
        const bool whole = w->k % 256 == 0;
        if constexpr (MT == 1) {
            const int64_t plane = DT == CQ_DTYPE_Q8_0 ? w->n * w->k : w->n * w->k / 2;
            if (m <= 32 && plane >= kOnceBytes)
                return whole ? launch_inst<DT, 1, false, true, false>(w, a, m, y, ksplit, d, s)
                             : launch_inst<DT, 1, false, true, true>(w, a, m, y, ksplit, d, s);
        }
        return whole ? launch_inst<DT, MT, false, false, false>(w, a, m, y, ksplit, d, s)
                     : launch_inst<DT, MT, false, false, true>(w, a, m, y, ksplit, d, s);
    }
}

template <int DT, int MT, bool DUMP> hipError_t launch_kh(const cq_weight *w, cq_act_view a, int64_t m, float *y, cq_mfma_dump d, hipStream_t s) {
    if (a.m_stride < (m + 32 * MT - 1) / (32 * MT) * (32 * MT)) return hipErrorInvalidValue;   // rows the last tile reads
    auto go = [&](auto sh, auto low) {
        constexpr bool SHORT = decltype(sh)::value, LOWER = decltype(low)::value;
        const size_t lds = TileKH<DT, MT>::kTotal;
        if (hipError_t e = cq_ensure_lds<gemm32_kh_kernel<DT, MT, DUMP, SHORT, LOWER>>(w->dev, lds); e != hipSuccess) return e;
        CQ_LAUNCH((gemm32_kh_kernel<DT, MT, DUMP, SHORT, LOWER>), dim3((unsigned)((w->n + 127) / 128), (unsigned)((m + MT * 32 - 1) / (MT * 32))), kThreads, lds, s, *w,
                  a, m, y, (int)cq_streams_result(w, m), d);
        return hipGetLastError();
    };
    auto whole_or_short = [&](auto low) {
        if constexpr (!DUMP)   // (whole K steps are all that is dumped)
            if (w->k % 256 != 0) return go(std::true_type{}, low);
        return go(std::false_type{}, low);
    };
    // One row of workgroups whose upper sixteen rows are padding (with 64-row tiles no faster).  An instance of its own: as a branch in the step, or
    // around two steps, the loop lost its unrolling or its registers (Q4_0 32003 x 3200 at 77 rows 42 -> 56 to 711 us).
    if constexpr (MT == 3)
        if (m <= 32 * MT - 16) return whole_or_short(std::true_type{});
    return whole_or_short(std::false_type{});
}
template <int DT, int CW, bool DUMP> hipError_t launch_few(const cq_weight *w, cq_act_view a, int64_t m, float *y, cq_mfma_dump d, hipStream_t s) {
    auto go = [&](auto on, auto sh) {
        constexpr bool ONCE = decltype(on)::value, SHORT = decltype(sh)::value;
        const size_t lds = Few<DT>::kTotal;
        if (hipError_t e = cq_ensure_lds<gemm32_few_kernel<DT, CW, DUMP, ONCE, SHORT>>(w->dev, lds); e != hipSuccess) return e;
        CQ_LAUNCH((gemm32_few_kernel<DT, CW, DUMP, ONCE, SHORT>), (unsigned)((w->n + 32 * CW - 1) / (32 * CW)), kThreads, lds, s, *w, a, m, y, d);
        return hipGetLastError();
    };
    if constexpr (!DUMP) {
        const bool once = (DT == CQ_DTYPE_Q8_0 ? w->n * w->k : w->n * w->k / 2) >= kOnceBytes;
        if (w->k % 256 != 0) return once ? go(std::true_type{}, std::true_type{}) : go(std::false_type{}, std::true_type{});
        if (once) return go(std::true_type{}, std::false_type{});
    }
    return go(std::false_type{}, std::false_type{});
}

template <int DT, bool DUMP> hipError_t launch_few_cw(const cq_weight *w, cq_act_view a, int64_t m, float *y, int cw, cq_mfma_dump d, hipStream_t s) {
    switch (cw) {
    case 1: return launch_few<DT, 1, DUMP>(w, a, m, y, d, s);
    case 2: return launch_few<DT, 2, DUMP>(w, a, m, y, d, s);
    case 4: return launch_few<DT, 4, DUMP>(w, a, m, y, d, s);
    default: return launch_few<DT, 8, DUMP>(w, a, m, y, d, s);
    }
}

template <int DT, bool DUMP>
hipError_t launch_dt(const cq_weight *w, cq_act_view a, int64_t m, float *y, bool y_cleared, cq_mfma_dump d, hipStream_t s) {
    const Plan p = pick_plan(w, m);
    if (p.few) return launch_few_cw<DT, DUMP>(w, a, m, y, p.few, d, s);
    if (p.kh) {
        if constexpr (kh_tallest<DT>() == 3)
            if (p.mt == 3) return launch_kh<DT, 3, DUMP>(w, a, m, y, d, s);
        return p.mt == 2 ? launch_kh<DT, 2, DUMP>(w, a, m, y, d, s) : launch_kh<DT, 1, DUMP>(w, a, m, y, d, s);
    }
    if (DUMP || w->k % 256 == 0) {   // (whole K steps are all that is dumped)
        if (p.tail == 2) return launch_tail<DT, 2, DUMP, false>(w, a, m, y, d, s);
        if (p.tail == 1) return launch_tail<DT, 1, DUMP, false>(w, a, m, y, d, s);
    } else if constexpr (!DUMP) {
        if (p.tail == 2) return launch_tail<DT, 2, false, true>(w, a, m, y, d, s);
        if (p.tail == 1) return launch_tail<DT, 1, false, true>(w, a, m, y, d, s);
    }
    if (p.mt == 1) return launch_mt<DT, 1, DUMP>(w, a, m, y, p.ksplit, y_cleared, d, s);
    if (p.mt == 2) return launch_mt<DT, 2, DUMP>(w, a, m, y, p.ksplit, y_cleared, d, s);
    return launch_mt<DT, 4, DUMP>(w, a, m, y, p.ksplit, y_cleared, d, s);
}

cq_grouped_plan pick_grouped(const cq_weight *w, const int32_t *offsets, int n_experts) {
    static constexpr cq_grouped_cost q8{5.8, 0.4, 1.15, 1.01, 0.97, 0.67}, q4{5.9, 0.85, 0.71, 1.16, 0.43, 0.69};
    return cq_plan_grouped_tiles(w, offsets, n_experts, w->dtype == CQ_DTYPE_Q8_0 ? q8 : q4);
}

template <int DT, int MT, bool SHORT>
hipError_t launch_grouped_mt(const cq_weight *const *experts, int n_experts, const int32_t *offsets, cq_act_view a, float *y,
                             int ksplit, bool y_cleared, hipStream_t s) {
    cq_group_args ga;
    const int tiles = cq_group_table(experts, n_experts, offsets, 32 * MT, &ga);
    if (tiles <= 0) return tiles == 0 ? hipSuccess : hipErrorInvalidConfiguration;
    const cq_weight *w = experts[0];
    const size_t lds = Tile<DT, MT>::kTotal;
    if (hipError_t e = cq_ensure_lds<gemm32_grouped_kernel<DT, MT, SHORT>>(w->dev, lds); e != hipSuccess) return e;
    if (ksplit > 1 && !y_cleared) {
        hipError_t e = cq_launch_fill_zero(y, (int64_t)offsets[n_experts] * w->n, s);
        if (e != hipSuccess) return e;
    }
    const dim3 grid((unsigned)((w->n + kWaves * 32 - 1) / (kWaves * 32)), (unsigned)tiles, (unsigned)ksplit);
    CQ_LAUNCH((gemm32_grouped_kernel<DT, MT, SHORT>), grid, kThreads, lds, s, ga, a, y, ksplit);
    return hipGetLastError();
}
template <int DT, bool SHORT>
hipError_t launch_grouped(const cq_weight *const *experts, int n_experts, const int32_t *offsets, cq_act_view a, float *y,
                          bool y_cleared, hipStream_t s) {
    const cq_grouped_plan p = pick_grouped(experts[0], offsets, n_experts);
    if (p.mt == 1) return launch_grouped_mt<DT, 1, SHORT>(experts, n_experts, offsets, a, y, p.ksplit, y_cleared, s);
    if (p.mt == 2) return launch_grouped_mt<DT, 2, SHORT>(experts, n_experts, offsets, a, y, p.ksplit, y_cleared, s);
    return launch_grouped_mt<DT, 4, SHORT>(experts, n_experts, offsets, a, y, p.ksplit, y_cleared, s);
}

}  // namespace

double cq_gemm32_grouped_us(const cq_weight *w, int n_experts, const int32_t *offsets) { return pick_grouped(w, offsets, n_experts).us; }
bool cq_gemm32_grouped_takes(const cq_weight *const *experts, int n_experts, const int32_t *offsets, int act_dtype) {
    return n_experts <= kMaxGroupExperts && cq_gemm32_takes(experts[0], act_dtype) && cq_group_tiles(offsets, n_experts, 32) <= kMaxGroupTiles;
}
bool cq_gemm32_grouped_splits_k(const cq_weight *const *experts, int n_experts, const int32_t *offsets) {
    return cq_group_tiles(offsets, n_experts, 32) > 0 && pick_grouped(experts[0], offsets, n_experts).ksplit > 1;
}
hipError_t cq_launch_gemm32_grouped(const cq_weight *const *experts, int n_experts, const int32_t *offsets, cq_act_view a, float *y,
                                    bool y_cleared, hipStream_t s) {
    if (a.m_stride < (int64_t)offsets[n_experts] + 127) return hipErrorInvalidValue;   // tiles of up to 128 rows from any row on
    const bool whole = experts[0]->k % 256 == 0;
    if (experts[0]->dtype == CQ_DTYPE_Q8_0)
        return whole ? launch_grouped<CQ_DTYPE_Q8_0, false>(experts, n_experts, offsets, a, y, y_cleared, s)
                     : launch_grouped<CQ_DTYPE_Q8_0, true>(experts, n_experts, offsets, a, y, y_cleared, s);
    return whole ? launch_grouped<CQ_DTYPE_Q4_0, false>(experts, n_experts, offsets, a, y, y_cleared, s)
                 : launch_grouped<CQ_DTYPE_Q4_0, true>(experts, n_experts, offsets, a, y, y_cleared, s);
}

bool cq_gemm32_takes(const cq_weight *w, int act_dtype) {
    // an even number of blocks per row, so that every row's scales begin on four bytes; the copies address 8 rows with 32-bit
    // offsets and may read up to 255 bytes past a plane's last row (weight planes: CQ_TAIL_PAD, activations: the next plane)
    return (w->dtype == CQ_DTYPE_Q8_0 || w->dtype == CQ_DTYPE_Q4_0) && act_dtype == CQ_DTYPE_Q8_0 && w->k >= 256 &&
           w->k % 64 == 0 && w->k <= (1 << 24) && w->n >= 32;
}
bool cq_gemm32_supported(const cq_weight *w, int act_dtype) {
    return cq_gemm32_takes(w, act_dtype) && w->k % 256 == 0 && w->n % 32 == 0;
}

// us of the tile launch beside the quantizer and the stores, from the plan's cost (fitted to the calls of groups_us in skinny.hip: 6 % rms).
double cq_gemm32_us(const cq_weight *w, int64_t m) {
    const Plan p = pick_plan(w, m);
    const int t = w->dtype == CQ_DTYPE_Q8_0 ? 0 : 1, form = p.few ? 2 : p.kh ? 1 : 0;
    static constexpr double start[2][3] = {{4.6, 3.25, 2.9}, {4.9, 3.7, 3.65}}, work[2][3] = {{0.97, 1.07, 1.30}, {0.92, 1.0, 1.16}};
    return start[t][form] + (work[t][form] * p.work + (t ? 1.13 : 1.33) * p.merge) / 16.0;
}
bool cq_gemm32_splits_k(const cq_weight *w, int64_t m) { return m > 0 && pick_plan(w, m).ksplit > 1; }

hipError_t cq_launch_gemm32(const cq_weight *w, cq_act_view a, int act_dtype, int64_t m, float *y, bool y_cleared,
                            hipStream_t s) {
    if (!cq_gemm32_takes(w, act_dtype)) return hipErrorNotSupported;
    if (m == 0) return hipSuccess;
    if (a.m_stride < (m <= 32 ? 32 : (m + 127) / 128 * 128)) return hipErrorInvalidValue;   // rows the last tile may read
    const cq_mfma_dump none{nullptr, nullptr};
    if (w->dtype == CQ_DTYPE_Q8_0) return launch_dt<CQ_DTYPE_Q8_0, false>(w, a, m, y, y_cleared, none, s);
    return launch_dt<CQ_DTYPE_Q4_0, false>(w, a, m, y, y_cleared, none, s);
}

hipError_t cq_launch_gemm32_dump(const cq_weight *w, cq_act_view a, int act_dtype, int64_t m, cq_mfma_dump d, hipStream_t s) {
    if (!cq_gemm32_supported(w, act_dtype)) return hipErrorNotSupported;
    if (m == 0) return hipSuccess;
    if (a.m_stride < (m <= 32 ? 32 : (m + 127) / 128 * 128)) return hipErrorInvalidValue;
    if (w->dtype == CQ_DTYPE_Q8_0) return launch_dt<CQ_DTYPE_Q8_0, true>(w, a, m, nullptr, true, d, s);
    return launch_dt<CQ_DTYPE_Q4_0, true>(w, a, m, nullptr, true, d, s);
}
