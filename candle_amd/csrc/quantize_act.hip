// Activation quantizers: f32 rows -> Q8_0 / Q8_1 / Q8K blocks, bit-identical to
// the reference's CPU code (candle-core/src/quantized/k_quants.rs):
//   BlockQ8_0::from_float :586-615     d = amax/127, id = 1/d, q = round(x*id) as i8
//   BlockQ8_1::from_float :665-691     as Q8_0 plus s = f16(f16(sum q) * d)
//   BlockQ8K::from_float  :1788-1825   signed max of the first largest |x|, iscale = -128/max,
//                                      q = min(127, round(iscale*x)) as i8, bsums, d = 1/iscale
// One wave (64 lanes) handles 256 consecutive elements of one row: lane l owns elements
// 4l..4l+3 (one float4 load, a whole 1 KiB line per wave).  Reductions are wave shuffles.
// Every f32 operation is a single IEEE operation in the reference's order (this file is
// compiled with -ffp-contract=off; `/` is correctly rounded).
//
// A step of the caller's model can run in front of the quantizer (cq_pre): silu(x) * x2 between the
// feed-forward projections (candle-transformers/src/models/quantized_llama.rs:56-63, silu as in
// candle-core/src/op.rs:607-609) is elementwise and goes into the kernels above; rms_norm
// (candle-nn/src/ops.rs:482-495: x / sqrt(mean(x^2) + eps) * alpha) needs the whole row first and
// has a kernel of its own with one workgroup per row.
#include "quantize_blocks.h"

#include <type_traits>

namespace {

__device__ __forceinline__ float silu_f(float v) { return v / (1.0f + expf(-v)); }
__device__ __forceinline__ float4 silu_mul4(float4 f, float4 a) {
    return make_float4(silu_f(f.x) * a.x, silu_f(f.y) * a.y, silu_f(f.z) * a.z, silu_f(f.w) * a.w);
}
__device__ __forceinline__ float4 rms_scale4(float4 f, float scale, float4 a) {
    return make_float4(scale * f.x * a.x, scale * f.y * a.y, scale * f.z * a.z, scale * f.w * a.w);
}

struct Sink {
    // GGML struct layout (AOS) or the workspace layout (qhip_internal.h)
    uint8_t *aos;
    cq_act_view v;
    cq_clear clear;
};

// The launch's threads share the floats to be cleared, four at a time (clear.p is 16-byte aligned).
__device__ __forceinline__ void clear_floats(const cq_clear &c) {
    if (!c.p) return;
    const int64_t step = (int64_t)gridDim.x * blockDim.x * 4;
    for (int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4; i < c.count; i += step) {
        if (i + 4 <= c.count) {
            *(float4 *)(c.p + i) = make_float4(0.f, 0.f, 0.f, 0.f);
        } else {
            for (int64_t j = i; j < c.count; j++) c.p[j] = 0.0f;
        }
    }
}

// a / b of non-negative numbers (a 64-bit division is a hundred vector instructions)
__device__ __forceinline__ int64_t divide(int64_t a, int64_t b) {
    return ((uint64_t)a | (uint64_t)b) >> 32 ? a / b : (int64_t)((uint32_t)a / (uint32_t)b);
}

// Q8_0 / Q8_1: eight 32-element blocks per wave, 8 lanes per block.  `f` = the lane's four values
// at element e0 of `row` (zeros in a lane past the end of the row); called by all 64 lanes.
template <bool AOS, bool Q8_1>
__device__ __forceinline__ void q8_0_chunk(const float4 f, bool active, int64_t row, int64_t e0, int64_t k, const Sink &out) {
    uint32_t packed;
    float d;
    int sum;
    cq_q8_0_of_eight(f, packed, d, sum);
    if (!active) return;
    const uint16_t dh = cq_f2h(d);
    const int64_t blk = row * (k / 32) + e0 / 32;
    const int within = (int)(e0 & 31);
    uint16_t sh = 0;
    if (Q8_1) sh = cq_f2h(cq_h2f(cq_f2h((float)sum)) * cq_h2f(dh));
    if (AOS) {
        const int ts = Q8_1 ? 36 : 34;
        uint8_t *b = out.aos + blk * ts;
        uint16_t *b16 = (uint16_t *)b;  // block offsets are even
        if (within == 0) {
            b16[0] = dh;
            if (Q8_1) b16[1] = sh;
        }
        uint16_t *q16 = (uint16_t *)(b + (Q8_1 ? 4 : 2) + within);
        q16[0] = (uint16_t)(packed & 0xffff);
        q16[1] = (uint16_t)(packed >> 16);
    } else {
        *(uint32_t *)(out.v.qs + row * k + e0) = packed;
        if (within == 0) {
            out.v.d[blk] = cq_h2f(dh);
            out.v.bsum32[blk] = (int16_t)sum;
            if (Q8_1) out.v.s16[blk] = sh;
            else out.v.dT[(e0 / 32) * out.v.m_stride + row] = cq_h2f(dh);
        }
    }
}

template <bool AOS, bool Q8_1, bool SILU>
__global__ void __launch_bounds__(256) quantize_q8_0_kernel(const float *__restrict__ x,
                                                            const int32_t *__restrict__ row_ids, int64_t m,
                                                            int64_t k, const float *__restrict__ x2, Sink out) {
    const int lane = threadIdx.x & 63;
    const int64_t chunks_per_row = (k + 255) / 256;
    const int64_t wave = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int64_t row = divide(wave, chunks_per_row);
    const int64_t e0 = (wave - row * chunks_per_row) * 256 + 4 * lane;
    const bool active = row < m && e0 < k;  // k % 32 == 0, so a lane is either fully inside or fully outside
    float4 f = make_float4(0.f, 0.f, 0.f, 0.f), f2 = f;
    if (active) {
        const int64_t src_row = row_ids ? (int64_t)row_ids[row] : row;
        f = *(const float4 *)(x + src_row * k + e0);
        if (SILU) f2 = *(const float4 *)(x2 + src_row * k + e0);
    }
    clear_floats(out.clear);   // (while the elements are on their way)
    if (row >= m) return;
    if (SILU && active) f = silu_mul4(f, f2);
    q8_0_chunk<AOS, Q8_1>(f, active, row, e0, k, out);
}

// Q8K: one 256-element block per wave.
// `f` = the lane's four values of block b_in_row of `row`; called by all 64 lanes.  SCALED: the
// block's scale is multiplied by `dscale` on the way out (the block then stands for dscale * f; a
// zero block if dscale is 0), which nothing before waits for.
template <bool AOS, bool SCALED = false>
__device__ __forceinline__ void q8k_chunk(const float4 f, int64_t row, int64_t b_in_row, int64_t k, const Sink &out,
                                          float dscale = 1.0f) {
    const int lane = threadIdx.x & 63;
    const int64_t blk = row * (k / 256) + b_in_row;

    uint32_t packed;
    int sum;   // lanes 4j .. 4j + 3 hold bsums[j]
    float d;
    cq_q8k_of_wave(f, lane, packed, d, sum);
    if (SCALED) {
        const bool zero = dscale == 0.0f;
        packed = zero ? 0u : packed;
        sum = zero ? 0 : sum;
        d = zero ? 0.0f : d * dscale;
    }
    if (AOS) {
        uint8_t *b = out.aos + blk * 292;  // 292 = 4 * 73: 4-byte aligned
        if (lane == 0) *(float *)b = d;
        *(uint32_t *)(b + 4 + 4 * lane) = packed;
        if ((lane & 3) == 0) *(int16_t *)(b + 260 + 2 * (lane >> 2)) = (int16_t)sum;
    } else {
        *(uint32_t *)(out.v.qs + row * k + b_in_row * 256 + 4 * lane) = packed;
        if (lane == 0) out.v.d[blk] = d;
        if ((lane & 3) == 0) out.v.bsums[blk * 16 + (lane >> 2)] = (int16_t)sum;
        // For the matrix-core kernels (block-major copies): d again, and for their min term the sixteen sums once more
        // as f16 (at most 16 * 128 in magnitude: exact), the operand of its contraction.
        const int64_t tb = b_in_row * out.v.m_stride + row;
        if (lane == 0) out.v.dT[tb] = d;
        if ((lane & 3) == 0) ((_Float16 *)out.v.bsh)[tb * 16 + (lane >> 2)] = (_Float16)(float)sum;
    }
}

// Many rows: a block per sixteen lanes, four blocks a wave.  Lane l of a block's sixteen holds elements 64i + 4l .. + 3 (i = 0..3),
// reductions end inside the sixteen lanes and every scalar step of a block (two divisions, stores) is shared by four.
// A wave a block (the kernel below) is bound by its vector instructions; here memory is.  Kernel
// alone, us, with a wave a block -> here: 512 x 4096 6.0 -> 3.3, 1024 x 4096 9.2 -> 5.7, 4096 x 4096 22.3 -> 15.4 (5.5 TB/s), with
// silu 32.9 -> 26.5, 4096 x 14336 123 -> 105.
template <bool AOS, bool SILU>
__global__ void __launch_bounds__(256) quantize_q8k_quad_kernel(const float *__restrict__ x, const int32_t *__restrict__ row_ids,
                                                                uint32_t blocks, uint32_t kb, const float *__restrict__ x2, Sink out) {
    if (blockIdx.x * 16 >= blocks) {   // (a workgroup that only clears)
        clear_floats(out.clear);
        return;
    }
    const uint32_t l = threadIdx.x & 15;
    const uint32_t blk = blockIdx.x * 16 + (threadIdx.x >> 4);
    const bool active = blk < blocks;
    const uint32_t at = active ? blk : blocks - 1;
    const uint32_t row = at / kb, b_in_row = at - row * kb;
    const int64_t k = (int64_t)kb * 256, src_row = row_ids ? (int64_t)row_ids[row] : row;
    const int64_t src = src_row * k + b_in_row * 256 + 4 * l;
    float4 f[4];
#pragma unroll
    for (int i = 0; i < 4; i++) f[i] = *(const float4 *)(x + src + 64 * i);
    clear_floats(out.clear);   // (while the elements are on their way)
    if (SILU) {
        float4 g[4];
#pragma unroll
        for (int i = 0; i < 4; i++) g[i] = *(const float4 *)(x2 + src + 64 * i);
#pragma unroll
        for (int i = 0; i < 4; i++) f[i] = silu_mul4(f[i], g[i]);
    }
    uint32_t packed[4];
    float d;
    int mine;
    cq_q8k_of_sixteen(f, (int)l, packed, d, mine);
    if (!active) return;
    // lane l stores bsums[4 * (l % 4) + l / 4]
    const uint32_t j = l & 3, sj = 4 * j + (l >> 2);
    if (AOS) {
        uint8_t *b = out.aos + (int64_t)blk * 292;   // 292 = 4 * 73: 4-byte aligned
        if (l == 0) *(float *)b = d;
#pragma unroll
        for (int i = 0; i < 4; i++) *(uint32_t *)(b + 4 + 64 * i + 4 * l) = packed[i];
        *(int16_t *)(b + 260 + 2 * sj) = (int16_t)mine;
    } else {
        int8_t *q = out.v.qs + (int64_t)blk * 256 + 4 * l;
#pragma unroll
        for (int i = 0; i < 4; i++) *(uint32_t *)(q + 64 * i) = packed[i];
        const int64_t tb = (int64_t)b_in_row * out.v.m_stride + row;
        if (l == 0) {
            out.v.d[blk] = d;
            out.v.dT[tb] = d;
        }
        out.v.bsums[(int64_t)blk * 16 + sj] = (int16_t)mine;
        ((_Float16 *)out.v.bsh)[tb * 16 + sj] = (_Float16)(float)mine;
    }
}

template <bool AOS, bool SILU>
__global__ void __launch_bounds__(256) quantize_q8k_kernel(const float *__restrict__ x,
                                                           const int32_t *__restrict__ row_ids, int64_t m, int64_t k,
                                                           const float *__restrict__ x2, Sink out) {
    const int lane = threadIdx.x & 63;
    const int64_t kb = k / 256;
    const int64_t blk = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int64_t row = divide(blk, kb);
    const int64_t b_in_row = blk - row * kb;
    float4 f = make_float4(0.f, 0.f, 0.f, 0.f), f2 = f;
    if (row < m) {
        const int64_t src_row = row_ids ? (int64_t)row_ids[row] : row;
        f = *(const float4 *)(x + src_row * k + b_in_row * 256 + 4 * lane);
        if (SILU) f2 = *(const float4 *)(x2 + src_row * k + b_in_row * 256 + 4 * lane);
    }
    clear_floats(out.clear);   // (while the elements are on their way)
    if (row >= m) return;
    if (SILU) f = silu_mul4(f, f2);
    q8k_chunk<AOS>(f, row, b_in_row, k, out);
}

// rms_norm in front of the quantizer: one workgroup per row.  The squares are added
// in a fixed order that does not depend on the kernel (the decode matvec's prologue follows it
// too, so a row gives the same bits whatever the batch): groups of 8 consecutive elements as two
// sequential sums of 4, added; a binary tree over the 32 groups of a 256-element chunk (group j
// with j^1, then ^2, ^4, ^8, ^16); then the chunks one after the other.  The reference's CPU code
// adds all squares one after the other: the two sums agree to rounding, not to the bit.
// scale = 1 / sqrt(mean + eps) multiplies the elements as in the reference's device kernel
// (candle-kernels/src/reduce.cu:161-172; its CPU code divides every element by the root).  The
// second pass:
//   Q8_0 / Q8_1: quantizes scale * x * alpha chunk by chunk;
//   Q8K: quantizes z = x * alpha and multiplies the block scales by `scale`: the quants of
//        scale * z are those of z, and the decode matvec uses the same form.
// ACT: 0 = Q8K, 1 = Q8_0, 2 = Q8_1.  Dynamic LDS: one float per chunk.
// A wave keeps its first kRmsHeld chunks (NW * kRmsHeld * 256 elements of the row) in registers between the two passes.
// Few rows are latency, and what a wave computes (about 400 instructions): sixteen waves of one row share the four vector
// units of a CU.  SPLIT: a row is spread over workgroups of kRmsSplit waves, each of which adds the squares of the whole row
// (from L2, four chunks side by side) and quantizes one chunk a wave; the same bits.  Kernel alone, us, one workgroup a row of
// sixteen waves -> split, 4 rows of Q8K: 4096 5.5 -> 4.5, 8192 8.3 -> 5.9, 16384 14.2 -> 8.4.  Up to 2048 elements the sixteen
// waves are as fast (3.7), and with more workgroups than CUs the second sum of the row costs more than it gives
// (64 rows of 8192: 8.4 against 8.8).  Eight waves a workgroup: 4096 5.2, 16384 7.6.
constexpr int kRmsHeld = 2, kRmsSplit = 4;
template <bool AOS, int ACT, int NW, bool SPLIT>
__global__ void __launch_bounds__(NW * 64) quantize_rms_rows_kernel(const float *__restrict__ x,
                                                                    const int32_t *__restrict__ row_ids, int64_t k,
                                                                    const float *__restrict__ alpha, float eps, Sink out) {
    extern __shared__ __align__(16) float chunk_sums[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int chunks = (int)((k + 255) / 256), parts = SPLIT ? (chunks + NW - 1) / NW : 1;
    const int64_t row = blockIdx.x / parts;
    const int part = (int)(blockIdx.x - row * parts);
    const int64_t src_row = row_ids ? (int64_t)row_ids[row] : row;
    const float *xr = x + src_row * k;
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    constexpr int kHeld = SPLIT ? 1 : kRmsHeld;
    float4 fx[kHeld], ax[kHeld];
#pragma unroll
    for (int i = 0; i < kHeld; i++) {
        const int64_t e0 = (int64_t)(wave + (SPLIT ? part : i) * NW) * 256 + 4 * lane;
        fx[i] = e0 < k ? *(const float4 *)(xr + e0) : zero;
        ax[i] = e0 < k ? *(const float4 *)(alpha + e0) : zero;
    }
    clear_floats(out.clear);
    // the sums of N chunks c, c + NW, ... (side by side: each is a chain of dependent additions)
    auto chunk_sums_of = [&](auto N, int c, const float4 *f) {
        float t[N], v = 0.0f;
#pragma unroll
        for (int i = 0; i < N; i++) {
            t[i] = f[i].x * f[i].x;
            t[i] += f[i].y * f[i].y;
            t[i] += f[i].z * f[i].z;
            t[i] += f[i].w * f[i].w;
        }
#pragma unroll
        for (int i = 0; i < N; i++) t[i] += dpp_f<kQuadSwap1>(t[i]);
#pragma unroll
        for (int i = 0; i < N; i++) t[i] += dpp_f<kQuadSwap2>(t[i]);
#pragma unroll
        for (int i = 0; i < N; i++) t[i] += dpp_f<kHalfMirror>(t[i]);
#pragma unroll
        for (int i = 0; i < N; i++) t[i] += dpp_f<kRowMirror>(t[i]);
#pragma unroll
        for (int i = 0; i < N; i++) {
            const float s = (readlane_f(t[i], 0) + readlane_f(t[i], 16)) + (readlane_f(t[i], 32) + readlane_f(t[i], 48));
            v = lane == i ? s : v;
        }
        if (lane < N && c + lane * NW < chunks) chunk_sums[c + lane * NW] = v;
    };
    // (zeros up to a multiple of 16 chunks: the sum below reads sixteen at a time)
    const int padded = (chunks + 15) / 16 * 16;
    if ((int)threadIdx.x < padded - chunks) chunk_sums[chunks + threadIdx.x] = 0.0f;
    constexpr std::integral_constant<int, SPLIT ? 4 : kHeld> at_once{};
    if constexpr (!SPLIT) chunk_sums_of(at_once, wave, fx);
    for (int c = SPLIT ? wave : wave + kHeld * NW; c < chunks; c += at_once * NW) {
        float4 f[at_once];
#pragma unroll
        for (int i = 0; i < at_once; i++) {
            const int64_t e0 = (int64_t)(c + i * NW) * 256 + 4 * lane;
            f[i] = e0 < k ? *(const float4 *)(xr + e0) : zero;
        }
        chunk_sums_of(at_once, c, f);
    }
    __syncthreads();
    float sum2 = 0.0f;
    for (int c = 0; c < padded; c += 16) {   // (sixteen reads in flight, the additions in order)
        float4 s4[4];
#pragma unroll
        for (int i = 0; i < 4; i++) s4[i] = *(const float4 *)(chunk_sums + c + 4 * i);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            sum2 += s4[i].x;
            sum2 += s4[i].y;
            sum2 += s4[i].z;
            sum2 += s4[i].w;
        }
    }
    const float scale = 1.0f / sqrtf(sum2 / (float)k + eps);
    // Q8K: a row whose scale is NaN, infinite or zero (NaN or infinities among its elements, squares that overflow) is
    // all NaN or all zero after the reference's normalisation and quantizes to zero blocks; z alone would not
    const float q8k_scale = scale > 0.0f && scale < __builtin_inff() ? scale : 0.0f;
    auto quantize = [&](int c, const float4 f, const float4 a) {
        const int64_t e0 = (int64_t)c * 256 + 4 * lane;
        if (ACT == 0) q8k_chunk<AOS, true>(make_float4(f.x * a.x, f.y * a.y, f.z * a.z, f.w * a.w), row, c, k, out, q8k_scale);
        else q8_0_chunk<AOS, ACT == 2>(rms_scale4(f, scale, a), e0 < k, row, e0, k, out);
    };
    if constexpr (SPLIT) {
        if (part * NW + wave < chunks) quantize(part * NW + wave, fx[0], ax[0]);
        return;
    }
#pragma unroll
    for (int i = 0; i < kHeld; i++)
        if (wave + i * NW < chunks) quantize(wave + i * NW, fx[i], ax[i]);
    for (int c = wave + kHeld * NW; c < chunks; c += NW) {
        const int64_t e0 = (int64_t)c * 256 + 4 * lane;
        const bool active = e0 < k;
        quantize(c, active ? *(const float4 *)(xr + e0) : zero, active ? *(const float4 *)(alpha + e0) : zero);
    }
}
template <bool AOS, int ACT>
void launch_rms(const float *x, const int32_t *row_ids, int64_t m, int64_t k, cq_pre pre, const Sink &out, hipStream_t s) {
    const int64_t chunks = (k + 255) / 256, parts = (chunks + kRmsSplit - 1) / kRmsSplit;
    const size_t lds = (size_t)(chunks + 15) / 16 * 64;
    if (chunks <= 4) quantize_rms_rows_kernel<AOS, ACT, 4, false><<<(unsigned)m, 256, lds, s>>>(x, row_ids, k, pre.aux, pre.eps, out);
    else if (chunks > 8 && m * parts <= cq_num_cus())
        quantize_rms_rows_kernel<AOS, ACT, kRmsSplit, true><<<(unsigned)(m * parts), kRmsSplit * 64, lds, s>>>(x, row_ids, k, pre.aux, pre.eps, out);
    else quantize_rms_rows_kernel<AOS, ACT, 16, false><<<(unsigned)m, 1024, lds, s>>>(x, row_ids, k, pre.aux, pre.eps, out);
}

// Blocks from which four share a wave: below, the chip is not full and the longer chain of a lane decides (256 rows of 1024: 2.8
// against 3.2 us; with silu, which is most of a lane's work, 64 rows of 1024 3.8 against 3.3).
constexpr int64_t kQuadBlocks = 1024;
template <bool AOS>
hipError_t launch(int act_dtype, const float *x, const int32_t *row_ids, int64_t m, int64_t k, cq_pre pre, Sink out,
                  hipStream_t s) {
    if (m == 0 || k == 0) return hipSuccess;
    if (act_dtype != CQ_DTYPE_Q8K && act_dtype != CQ_DTYPE_Q8_0 && act_dtype != CQ_DTYPE_Q8_1) return hipErrorInvalidValue;
    const int threads = 256, waves = threads / 64;
    if (pre.kind == CQ_PRE_RMS_NORM) {
        if ((size_t)((k + 255) / 256) * 4 > 48 * 1024) return hipErrorInvalidValue;   // rows of more than 3 million elements
        if (act_dtype == CQ_DTYPE_Q8K) launch_rms<AOS, 0>(x, row_ids, m, k, pre, out, s);
        else if (act_dtype == CQ_DTYPE_Q8_0) launch_rms<AOS, 1>(x, row_ids, m, k, pre, out, s);
        else launch_rms<AOS, 2>(x, row_ids, m, k, pre, out, s);
        return hipGetLastError();
    }
    const bool silu = pre.kind == CQ_PRE_SILU_MUL;
    const int64_t nw = act_dtype == CQ_DTYPE_Q8K ? m * (k / 256) : m * ((k + 255) / 256);
    // (workgroups past the last block only clear: 21 rows on 14336 weight rows clear 1.2 MB beside 84 workgroups of work)
    const int64_t clearers = out.clear.p ? (out.clear.count + 4 * threads - 1) / (4 * threads) : 0;
    const int64_t least = clearers < 2 * cq_num_cus() ? clearers : 2 * cq_num_cus(), need = (nw + waves - 1) / waves;
    const unsigned grid = (unsigned)(need > least ? need : least);
    if (act_dtype == CQ_DTYPE_Q8K && nw >= kQuadBlocks && nw < (1ll << 31)) {
        const unsigned quads = (unsigned)((nw + 15) / 16 > least ? (nw + 15) / 16 : least);
        if (silu) quantize_q8k_quad_kernel<AOS, true><<<quads, threads, 0, s>>>(x, row_ids, (uint32_t)nw, (uint32_t)(k / 256), pre.aux, out);
        else quantize_q8k_quad_kernel<AOS, false><<<quads, threads, 0, s>>>(x, row_ids, (uint32_t)nw, (uint32_t)(k / 256), nullptr, out);
    } else if (act_dtype == CQ_DTYPE_Q8K) {
        if (silu) quantize_q8k_kernel<AOS, true><<<grid, threads, 0, s>>>(x, row_ids, m, k, pre.aux, out);
        else quantize_q8k_kernel<AOS, false><<<grid, threads, 0, s>>>(x, row_ids, m, k, nullptr, out);
    } else if (act_dtype == CQ_DTYPE_Q8_0) {
        if (silu) quantize_q8_0_kernel<AOS, false, true><<<grid, threads, 0, s>>>(x, row_ids, m, k, pre.aux, out);
        else quantize_q8_0_kernel<AOS, false, false><<<grid, threads, 0, s>>>(x, row_ids, m, k, nullptr, out);
    } else {
        if (silu) quantize_q8_0_kernel<AOS, true, true><<<grid, threads, 0, s>>>(x, row_ids, m, k, pre.aux, out);
        else quantize_q8_0_kernel<AOS, true, false><<<grid, threads, 0, s>>>(x, row_ids, m, k, nullptr, out);
    }
    return hipGetLastError();
}

}  // namespace

hipError_t cq_launch_quantize_act_aos(int act_dtype, const float *x, int64_t m, int64_t k, cq_pre pre, void *dst,
                                      hipStream_t s) {
    Sink out{};
    out.aos = (uint8_t *)dst;
    return launch<true>(act_dtype, x, nullptr, m, k, pre, out, s);
}

hipError_t cq_launch_quantize_act_ws(int act_dtype, const float *x, const int32_t *row_ids, int64_t m, int64_t k,
                                     cq_pre pre, cq_act_view v, cq_clear clear, hipStream_t s) {
    Sink out{};
    out.v = v;
    out.clear = clear;
    return launch<false>(act_dtype, x, row_ids, m, k, pre, out, s);
}
