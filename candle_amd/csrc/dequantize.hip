// Device planes -> f32 / f16 (QTensor::dequantize, dequantize_f16;
// candle-core/src/quantized/mod.rs:361-382, CUDA precedent cuda.rs:69-181).
// The f32 values are those of T::to_float (k_quants.rs:163-183, :329-349, :533-558, :568-584, :841-872, :1094-1146, :1313-1341,
// :1527-1564, :1716-1746): same products in the same order, no contraction.  The f16 output is the
// f32 output rounded to nearest-even, as the reference's tests require
// (candle-core/tests/quantized_tests.rs:229-234).
// One thread per 16-byte lane of the main plane; a wave covers 1 KiB of it and one run of the output.
#include "qhip_internal.h"

namespace {

constexpr int kThreads = 256;

// The results of a wave's 64 threads (ELEMS each) are one run of the output, of which a thread holds sixteen consecutive elements here and
// there: they go through LDS, so that every store of the wave is a whole KiB in lane order.  Bound: HBM.  Straight from the threads a store
// instruction touches every line of the run and fills a quarter of it (f16: half).  Kernel times, us, from the threads -> through LDS: f16 Q6K
// 32000 x 4096 70.7 -> 63.3, Q4K 11008 x 4096 20.9 -> 18.1, Q4_0 8192 x 4096 24.8 -> 14.0; f32 Q6K 163 -> 105, Q4K 56.2 -> 30.9, Q4_0 43.1 -> 23.5,
// Q8_0 43.7 -> 25.7.  STREAM: stores marked non-temporal (kStreamBytes says when); marking the reads so costs 5-20 %.
template <bool F16, bool STREAM, int ELEMS> struct Run {
    static constexpr int kSize = F16 ? 2 : 4, kBytes = 64 * ELEMS * kSize, kPer16 = 16 / kSize;
    uint8_t *lds;   // this wave's kBytes
    __device__ __forceinline__ static uint8_t *of_wave() {
        __shared__ __align__(16) uint8_t img[kThreads / 64 * kBytes];
        return img + threadIdx.x / 64 * kBytes;
    }
    // chunk c of 16 bytes sits at c ^ (c / 16 % 16): the sixteen lanes that LDS serves at a time meet no bank twice, on either side
    __device__ __forceinline__ static uint32_t at(uint32_t c) { return (c ^ (c >> 4 & 15)) * 16; }
    // sixteen consecutive results starting at element i of the run (a multiple of 16)
    __device__ __forceinline__ void put(int i, const float (&v)[16]) const {
        const uint32_t c = (uint32_t)i / kPer16;
        if (F16) {
            uint32_t w[8];
#pragma unroll
            for (int j = 0; j < 8; j++) w[j] = (uint32_t)cq_f2h(v[2 * j]) | ((uint32_t)cq_f2h(v[2 * j + 1]) << 16);
            *(uint4 *)(lds + at(c)) = make_uint4(w[0], w[1], w[2], w[3]);
            *(uint4 *)(lds + at(c + 1)) = make_uint4(w[4], w[5], w[6], w[7]);
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) *(float4 *)(lds + at(c + j)) = make_float4(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
        }
    }
    // the run's elements first .. (as far as `total` goes) to the output
    __device__ __forceinline__ void store(float *d32, uint16_t *d16, int64_t first, int64_t total) const {
        // the other lanes' writes: the hardware carries out a wave's LDS operations in order, the fences keep the compiler to it
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        typedef uint32_t u4 __attribute__((ext_vector_type(4)));
        u4 *dst = (u4 *)(F16 ? (void *)(d16 + first) : (void *)(d32 + first));
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int j = 0; j < kBytes / 1024; j++) {
            const uint32_t c = j * 64 + lane;
            const u4 v = *(const u4 *)(lds + at(c));
            if (first + (int64_t)c * kPer16 < total) {
                if constexpr (STREAM) __builtin_nontemporal_store(v, dst + c);
                else dst[c] = v;
            }
        }
    }
};

template <bool F16, bool STREAM>
__global__ void dequant_q4_0(const uint8_t *__restrict__ qs, const uint16_t *__restrict__ dpl, int64_t nblocks,
                             float *d32, uint16_t *d16) {
    const Run<F16, STREAM, 32> run{Run<F16, STREAM, 32>::of_wave()};
    const int64_t t = (int64_t)blockIdx.x * kThreads + threadIdx.x, b = t < nblocks ? t : nblocks - 1;
    const uint4 q = *(const uint4 *)(qs + b * 16);
    const float d = cq_h2f(dpl[b]);
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
    float lo[16], hi[16];
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const uint32_t byte = (w[j >> 2] >> (8 * (j & 3))) & 0xff;
        const int x0 = (int)(byte & 0xF) - 8, x1 = (int)(byte >> 4) - 8;
        lo[j] = (float)x0 * d;
        hi[j] = (float)x1 * d;
    }
    const int lane = threadIdx.x & 63;
    run.put(lane * 32, lo);
    run.put(lane * 32 + 16, hi);
    run.store(d32, d16, (t - lane) * 32, nblocks * 32);
}

// MIN: Q4_1 / Q5_1 held as Q8_0 planes plus the plane of block minima: q * d + m (k_quants.rs:329-349, :533-558)
template <bool F16, bool STREAM, bool MIN>
__global__ void dequant_q8_0(const uint8_t *__restrict__ qs, const uint16_t *__restrict__ dpl,
                             const uint16_t *__restrict__ mpl, int64_t nunits, float *d32, uint16_t *d16) {
    const Run<F16, STREAM, 16> run{Run<F16, STREAM, 16>::of_wave()};
    const int64_t t = (int64_t)blockIdx.x * kThreads + threadIdx.x, u = t < nunits ? t : nunits - 1;  // 16 elements each
    const uint4 q = *(const uint4 *)(qs + u * 16);
    const float d = cq_h2f(dpl[u >> 1]);
    const float mn = MIN ? cq_h2f(mpl[u >> 1]) : 0.0f;
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
    float out[16];
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const int8_t v = (int8_t)((w[j >> 2] >> (8 * (j & 3))) & 0xff);
        out[j] = (float)v * d;
        if (MIN) out[j] = out[j] + mn;
    }
    const int lane = threadIdx.x & 63;
    run.put(lane * 16, out);
    run.store(d32, d16, (t - lane) * 16, nunits * 16);
}

// Q5 (Q5K, to_float k_quants.rs:1527-1564): the fifth bits come from the re-ordered qh plane, words
// {L, H} per 32 qs bytes, bit 8c + i for byte c of qs word i.
template <bool F16, bool STREAM, bool Q5>
__global__ void dequant_q4k(const uint8_t *__restrict__ qs, const uint8_t *__restrict__ hd,
                            const uint8_t *__restrict__ qh, int64_t nunits, float *d32, uint16_t *d16) {
    const Run<F16, STREAM, 32> run{Run<F16, STREAM, 32>::of_wave()};
    const int64_t t = (int64_t)blockIdx.x * kThreads + threadIdx.x, u = t < nunits ? t : nunits - 1;  // 16 bytes of qs = 32 elements
    const int64_t b = u >> 3;
    const int p = (int)(u & 7), g = p >> 1, half = p & 1;
    const uint4 q = *(const uint4 *)(qs + u * 16);
    const uint32_t *h = (const uint32_t *)(hd + b * CQ_Q4K_HDR);
    const uint32_t dd = h[0], rec = h[1 + g];
    const float d = cq_h2f((uint16_t)(dd & 0xffff)), dmin = cq_h2f((uint16_t)(dd >> 16));
    const int sc1 = (int)(rec & 0xff), sc2 = (int)((rec >> 8) & 0xff);
    const int m1 = (int)((rec >> 16) & 0xff), m2 = (int)(rec >> 24);
    const float d1 = d * (float)sc1, mm1 = dmin * (float)m1;
    const float d2 = d * (float)sc2, mm2 = dmin * (float)m2;
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
    const int lane = threadIdx.x & 63, base = (lane >> 3) * 256 + 64 * g + 16 * half;   // (of the run; past the end nothing is stored)
    uint2 fifth = make_uint2(0u, 0u);
    if (Q5) fifth = *(const uint2 *)(qh + (b * 4 + g) * 8);
    float lo[16], hi[16];
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const uint32_t byte = (w[j >> 2] >> (8 * (j & 3))) & 0xff;
        const int bit = 8 * (j & 3) + 4 * half + (j >> 2);
        lo[j] = d1 * (float)((byte & 0xF) + (((fifth.x >> bit) & 1u) << 4)) - mm1;
        hi[j] = d2 * (float)((byte >> 4) + (((fifth.y >> bit) & 1u) << 4)) - mm2;
    }
    run.put(base, lo);
    run.put(base + 32, hi);
    run.store(d32, d16, (t - lane) * 32, nunits * 32);
}

// MIN: Q2K held as Q6K planes plus the groups' minima and dmin: (d * sc) * q - dmin * m (k_quants.rs:841-872)
template <bool F16, bool STREAM, bool MIN>
__global__ void dequant_q6k(const uint8_t *__restrict__ ql, const uint8_t *__restrict__ qh,
                            const int8_t *__restrict__ sc, const uint16_t *__restrict__ dpl,
                            const uint8_t *__restrict__ mins, const uint16_t *__restrict__ dmins, int64_t nunits,
                            float *d32, uint16_t *d16) {
    const Run<F16, STREAM, 32> run{Run<F16, STREAM, 32>::of_wave()};
    const int64_t thread = (int64_t)blockIdx.x * kThreads + threadIdx.x, u = thread < nunits ? thread : nunits - 1;  // 16 bytes of ql = 32 elements
    const int64_t b = u >> 3;
    const int p = (int)(u & 7), h = p >> 2, t = (p >> 1) & 1, i0 = (p & 1) * 16;
    const uint4 q = *(const uint4 *)(ql + u * 16);
    const uint2 hh = *(const uint2 *)(qh + u * 8);
    const float d = cq_h2f(dpl[b]);
    // low nibbles: elements 128h + 32t + i0 + e, one 16-element scale group; high nibbles: +64
    const float s_lo = (float)sc[u * 2], s_hi = (float)sc[u * 2 + 1];  // re-packed: the lane's two scales
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
    const uint32_t hw[2] = {hh.x, hh.y};
    const int lane = threadIdx.x & 63, base = (lane >> 3) * 256 + 128 * h + 32 * t + i0;   // (of the run; past the end nothing is stored)
    float lo[16], hi[16];
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const int wi = e >> 2, c = e & 3;
        const uint32_t byte = (w[wi] >> (8 * c)) & 0xff;
        const uint32_t hb = (hw[wi >> 1] >> (8 * c)) & 0xff;
        const int sh = (wi & 1) * 4;
        const int q_lo = (int)((byte & 0xF) | (((hb >> sh) & 3) << 4)) - 32;
        const int q_hi = (int)((byte >> 4) | (((hb >> (sh + 2)) & 3) << 4)) - 32;
        lo[e] = d * s_lo * (float)q_lo;
        hi[e] = d * s_hi * (float)q_hi;
    }
    if (MIN) {
        // the lane's low-nibble elements are group 8h + 2t + p%2 of the block, the high-nibble ones four groups on
        const int j = 8 * h + 2 * t + (p & 1);
        const float dmin = cq_h2f(dmins[b]);
        const float ml_lo = dmin * (float)mins[b * 16 + j], ml_hi = dmin * (float)mins[b * 16 + j + 4];
#pragma unroll
        for (int e = 0; e < 16; e++) {
            lo[e] = lo[e] - ml_lo;
            hi[e] = hi[e] - ml_hi;
        }
    }
    run.put(base, lo);
    run.put(base + 64, hi);
    run.store(d32, d16, (thread - lane) * 32, nunits * 32);
}

template <bool F16, bool STREAM>
hipError_t launch(const cq_weight *w, float *d32, uint16_t *d16, hipStream_t s) {
    const int threads = kThreads;
    const int64_t total = w->n * w->k;
    if (total == 0) return hipSuccess;
    auto grid = [&](int64_t n) { return (unsigned)((n + threads - 1) / threads); };
    switch (w->dtype) {
    case CQ_DTYPE_Q4_0:
        dequant_q4_0<F16, STREAM><<<grid(total / 32), threads, 0, s>>>(w->p0, (const uint16_t *)w->p1, total / 32, d32, d16);
        break;
    case CQ_DTYPE_Q8_0:
        if (cq_has_min32(w->ggml_dtype))
            dequant_q8_0<F16, STREAM, true><<<grid(total / 16), threads, 0, s>>>(w->p0, (const uint16_t *)w->p1, (const uint16_t *)w->p2,
                                                                                 total / 16, d32, d16);
        else
            dequant_q8_0<F16, STREAM, false><<<grid(total / 16), threads, 0, s>>>(w->p0, (const uint16_t *)w->p1, nullptr, total / 16, d32, d16);
        break;
    case CQ_DTYPE_Q4K:
        dequant_q4k<F16, STREAM, false><<<grid(total / 32), threads, 0, s>>>(w->p0, w->p1, nullptr, total / 32, d32, d16);
        break;
    case CQ_DTYPE_Q5K:
        dequant_q4k<F16, STREAM, true><<<grid(total / 32), threads, 0, s>>>(w->p0, w->p1, w->p2, total / 32, d32, d16);
        break;
    case CQ_DTYPE_Q6K:
        if (cq_has_min16(w->ggml_dtype))
            dequant_q6k<F16, STREAM, true><<<grid(total / 32), threads, 0, s>>>(w->p0, w->p1, (const int8_t *)w->p2, (const uint16_t *)w->p3,
                                                                                w->p4, (const uint16_t *)w->p5, total / 32, d32, d16);
        else
            dequant_q6k<F16, STREAM, false><<<grid(total / 32), threads, 0, s>>>(w->p0, w->p1, (const int8_t *)w->p2, (const uint16_t *)w->p3,
                                                                                 nullptr, nullptr, total / 32, d32, d16);
        break;
    case CQ_DTYPE_Q8K: return cq_launch_dequantize_q8k(w, d32, d16, s);
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// Outputs of more bytes are stored non-temporal.  What reads a dequantized tensor next finds it in the 256 MB of cache in front of the HBM, as long
// as it did not push itself out.  Dequantize and a product of sixteen rows with the result (torch), us, plain / non-temporal: f16 Q4K 512 x 1024
// 8.0/9.7, 4096 x 4096 28.1/30.7, 20480 x 4096 (168 MB) 74.5/94.2, 24576 (201 MB) 77.8/90.8, 28672 (235 MB) 120.4/117.3, 32000 (262 MB) 119.8/116.4,
// 64000 x 2048 108.0/116.3, 40960 x 4096 (336 MB) 164.5/146.3; f32 Q6K 8192 x 8192 (268 MB) 100.5/110.2, 20480 x 4096 (336 MB) 153.1/138.6.  235 to 268
// MB are level over six shapes and three types.  Without a reader plain is behind by up to 30 % at 8 to 33 MB, level from there to 201 MB (f16 Q6K
// 20480 x 4096 40.4/41.8) and 5 % behind beyond (32000 x 4096 68.5/63.9).
constexpr int64_t kStreamBytes = 240000000;

}  // namespace

hipError_t cq_launch_dequantize(const cq_weight *w, float *dst32, uint16_t *dst16, hipStream_t s) {
    const bool stream = w->n * w->k * (dst16 ? 2 : 4) > kStreamBytes;
    if (dst16) return stream ? launch<true, true>(w, nullptr, dst16, s) : launch<true, false>(w, nullptr, dst16, s);
    return stream ? launch<false, true>(w, dst32, nullptr, s) : launch<false, false>(w, dst32, nullptr, s);
}
