// GGML array-of-blocks <-> device planes (and back).  Pure byte permutations (repack_units.h):
// cq_launch_unpack(cq_launch_repack(x)) == x for every input.
//
// Replaces the plain host->device copy of cuda::load_quantized
// (candle-core/src/quantized/cuda.rs:591-612); the inverse serves QStorage::data
// (mod.rs:118-130).
#include "repack_units.h"

namespace {

template <int DT> __global__ void __launch_bounds__(256) repack_kernel(const uint8_t *__restrict__ aos, cq_planes pl, int64_t nblocks) {
    constexpr int U = Ggml<DT>::kUnits;
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, b = t / U;
    if (b < nblocks) repack_unit<DT, false>((uint8_t *)aos + b * Ggml<DT>::kSize, b, (int)(t - b * U), pl);
}

// Blocks first .. first + nblocks - 1 to `out`, which may be pinned host memory: the blocks are put together in LDS and leave in runs of
// 16-byte stores, whatever their size.
template <int DT> struct UnpackGroup { static constexpr int kBlocks = Ggml<DT>::kUnits == 1 ? 256 : 64; };
template <int DT> __global__ void __launch_bounds__(256) unpack_kernel(cq_planes pl, int64_t first, int64_t nblocks, uint8_t *__restrict__ out) {
    constexpr int U = Ggml<DT>::kUnits, TS = Ggml<DT>::kSize, PER = UnpackGroup<DT>::kBlocks;
    static_assert(PER * TS % 16 == 0, "whole 16-byte groups");
    __shared__ __align__(16) uint8_t img[PER * TS];
    const int64_t g0 = (int64_t)blockIdx.x * PER;
    const int count = (int)(nblocks - g0 < PER ? nblocks - g0 : PER);
    for (int i = threadIdx.x; i < count * U; i += 256) repack_unit<DT, true>(img + i / U * TS, first + g0 + i / U, i % U, pl);
    __syncthreads();
    uint8_t *dst = out + g0 * TS;
    const int whole = count * TS / 16;
    for (int i = threadIdx.x; i < whole; i += 256) ((uint4 *)dst)[i] = ((const uint4 *)img)[i];
    for (int i = whole * 8 + threadIdx.x; i < count * TS / 2; i += 256) ((uint16_t *)dst)[i] = ((const uint16_t *)img)[i];
}

// The allocation as all-zero GGML blocks leave it: planes 0, 1 and 2 (16-byte groups up to their ends) of one byte each, zeros elsewhere.
__global__ void __launch_bounds__(256) zero_planes_kernel(uint4 *__restrict__ base, int64_t groups, int64_t end0, int64_t from1, int64_t end1,
                                                          int64_t from2, int64_t end2, uint32_t v0, uint32_t v1, uint32_t v2) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= groups) return;
    const uint32_t v = i < end0 ? v0 : i >= from1 && i < end1 ? v1 : i >= from2 && i < end2 ? v2 : 0u;
    base[i] = make_uint4(v, v, v, v);
}

cq_planes planes_of(const cq_weight *w) { return cq_planes{w->p0, w->p1, w->p2, w->p3, w->p4, w->p5}; }

template <int DT> hipError_t repack(const cq_weight *w, const uint8_t *aos, int64_t nblocks, hipStream_t s) {
    hipLaunchKernelGGL(repack_kernel<DT>, dim3((unsigned)((nblocks * Ggml<DT>::kUnits + 255) / 256)), dim3(256), 0, s, aos, planes_of(w), nblocks);
    return hipGetLastError();
}
template <int DT> hipError_t unpack(const cq_weight *w, int64_t first, int64_t nblocks, uint8_t *out, hipStream_t s) {
    constexpr int PER = UnpackGroup<DT>::kBlocks;
    hipLaunchKernelGGL(unpack_kernel<DT>, dim3((unsigned)((nblocks + PER - 1) / PER)), dim3(256), 0, s, planes_of(w), first, nblocks, out);
    return hipGetLastError();
}

}  // namespace

hipError_t cq_launch_zero_planes(const cq_weight *w, hipStream_t s) {
    const int64_t groups = (int64_t)(w->alloc_bytes / 16), from1 = (w->p1 - w->p0) / 16, from2 = (w->p2 - w->p0) / 16, elems = w->n * w->k;
    int64_t g0 = 0, g1 = 0, g2 = 0;   // 16-byte groups of the planes
    uint32_t v0 = 0, v1 = 0, v2 = 0;
    switch (w->ggml_dtype) {
    case CQ_DTYPE_Q5_0: g0 = elems / 16; v0 = 0xf0f0f0f0u; break;                             // q - 16
    case CQ_DTYPE_Q3K:                                                                        // six-bit quants q + 28, scales -32
        g0 = elems / 32; v0 = 0xccccccccu;
        g1 = elems / 64; v1 = 0x55555555u;
        g2 = elems / 256; v2 = 0xe0e0e0e0u;
        break;
    case CQ_DTYPE_Q2K: g1 = elems / 64; v1 = 0xaaaaaaaau; break;                              // six-bit quants q + 32
    default: break;
    }
    if (groups == 0) return hipSuccess;
    hipLaunchKernelGGL(zero_planes_kernel, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, s, (uint4 *)w->base, groups, g0, from1, from1 + g1,
                       from2, from2 + g2, v0, v1, v2);
    return hipGetLastError();
}

hipError_t cq_launch_repack(const cq_weight *w, const uint8_t *aos_dev, hipStream_t s) {
    const int64_t nb = w->n * (w->k / cq_block_size(w->dtype));
    if (nb == 0) return hipSuccess;
    switch (w->ggml_dtype) {
    case CQ_DTYPE_Q4_0: return repack<CQ_DTYPE_Q4_0>(w, aos_dev, nb, s);
    case CQ_DTYPE_Q4_1: return repack<CQ_DTYPE_Q4_1>(w, aos_dev, nb, s);
    case CQ_DTYPE_Q5_0: return repack<CQ_DTYPE_Q5_0>(w, aos_dev, nb, s);
    case CQ_DTYPE_Q5_1: return repack<CQ_DTYPE_Q5_1>(w, aos_dev, nb, s);
    case CQ_DTYPE_Q8_0: return repack<CQ_DTYPE_Q8_0>(w, aos_dev, nb, s);
    case CQ_DTYPE_Q2K: return repack<CQ_DTYPE_Q2K>(w, aos_dev, nb, s);
    case CQ_DTYPE_Q3K: return repack<CQ_DTYPE_Q3K>(w, aos_dev, nb, s);
    case CQ_DTYPE_Q4K: return repack<CQ_DTYPE_Q4K>(w, aos_dev, nb, s);
    case CQ_DTYPE_Q5K: return repack<CQ_DTYPE_Q5K>(w, aos_dev, nb, s);
    case CQ_DTYPE_Q6K: return repack<CQ_DTYPE_Q6K>(w, aos_dev, nb, s);
    case CQ_DTYPE_Q8K: return cq_launch_repack_q8k(w, (uint8_t *)aos_dev, false, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t cq_launch_unpack(const cq_weight *w, int64_t first, int64_t nblocks, uint8_t *aos, hipStream_t s) {
    if (nblocks == 0) return hipSuccess;
    switch (w->ggml_dtype) {
    case CQ_DTYPE_Q4_0: return unpack<CQ_DTYPE_Q4_0>(w, first, nblocks, aos, s);
    case CQ_DTYPE_Q4_1: return unpack<CQ_DTYPE_Q4_1>(w, first, nblocks, aos, s);
    case CQ_DTYPE_Q5_0: return unpack<CQ_DTYPE_Q5_0>(w, first, nblocks, aos, s);
    case CQ_DTYPE_Q5_1: return unpack<CQ_DTYPE_Q5_1>(w, first, nblocks, aos, s);
    case CQ_DTYPE_Q8_0: return unpack<CQ_DTYPE_Q8_0>(w, first, nblocks, aos, s);
    case CQ_DTYPE_Q2K: return unpack<CQ_DTYPE_Q2K>(w, first, nblocks, aos, s);
    case CQ_DTYPE_Q3K: return unpack<CQ_DTYPE_Q3K>(w, first, nblocks, aos, s);
    case CQ_DTYPE_Q4K: return unpack<CQ_DTYPE_Q4K>(w, first, nblocks, aos, s);
    case CQ_DTYPE_Q5K: return unpack<CQ_DTYPE_Q5K>(w, first, nblocks, aos, s);
    case CQ_DTYPE_Q6K: return unpack<CQ_DTYPE_Q6K>(w, first, nblocks, aos, s);
    case CQ_DTYPE_Q8K: return first == 0 ? cq_launch_repack_q8k(w, aos, true, s) : hipErrorInvalidValue;   // (all blocks)
    default: return hipErrorInvalidValue;
    }
}
