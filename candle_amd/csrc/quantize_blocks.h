// The arithmetic of the activation quantizers, shared by the quantizer launches (quantize_act.hip) and the small-batch kernels that
// quantize their rows themselves (skinny.hip): the same operations in the same order, so the same bytes from either.
#pragma once
#include "qhip_internal.h"

#if defined(__HIPCC__)
// Q8K (k_quants.rs:1788-1825): a block per sixteen lanes.  Lane l of a block's sixteen holds elements 64i + 4l .. + 3 (i = 0..3) in `f`; on
// return the quants of those elements, four a word, the block scale, and of the block's sums of sixteen the one with index
// 4 * (l % 4) + l / 4.
// The signed extremes replace the search for the first largest |x|: only where both signs reach it does the position decide.
__device__ __forceinline__ void cq_q8k_of_sixteen(const float4 (&f)[4], int l, uint32_t (&packed)[4], float &d, int &bsum) {
    float hi = 0.0f, lo = 0.0f;   // (NaN elements fall out of both)
#pragma unroll
    for (int i = 0; i < 4; i++) {
        hi = fmaxf(fmaxf(fmaxf(fmaxf(hi, f[i].x), f[i].y), f[i].z), f[i].w);
        lo = fminf(fminf(fminf(fminf(lo, f[i].x), f[i].y), f[i].z), f[i].w);
    }
    hi = fmaxf(hi, dpp_f<kQuadSwap1>(hi));
    lo = fminf(lo, dpp_f<kQuadSwap1>(lo));
    hi = fmaxf(hi, dpp_f<kQuadSwap2>(hi));
    lo = fminf(lo, dpp_f<kQuadSwap2>(lo));
    hi = fmaxf(hi, dpp_f<kHalfMirror>(hi));
    lo = fminf(lo, dpp_f<kHalfMirror>(lo));
    hi = fmaxf(hi, dpp_f<kRowMirror>(hi));
    lo = fminf(lo, dpp_f<kRowMirror>(lo));
    const float amax = fmaxf(hi, -lo);
    float max = hi > -lo ? hi : lo;
    if (__any(hi == -lo && amax != 0.0f)) {   // both signs: the sign of the first of them
        int idx = 0x7fffffff;
#pragma unroll
        for (int i = 3; i >= 0; i--) {
            const float v[4] = {f[i].x, f[i].y, f[i].z, f[i].w};
#pragma unroll
            for (int c = 3; c >= 0; c--)
                if (fabsf(v[c]) == amax) idx = 2 * (64 * i + 4 * l + c) + (v[c] < 0.0f ? 1 : 0);
        }
        idx = min(idx, dpp_i<kQuadSwap1>(idx));
        idx = min(idx, dpp_i<kQuadSwap2>(idx));
        idx = min(idx, dpp_i<kHalfMirror>(idx));
        idx = min(idx, dpp_i<kRowMirror>(idx));
        if (hi == -lo) max = idx & 1 ? lo : hi;
    }
    const bool any = amax != 0.0f;
    const float iscale = -128.0f / max;
    d = any ? 1.0f / iscale : 0.0f;
    int sum[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float v[4] = {f[i].x, f[i].y, f[i].z, f[i].w};
        uint32_t q[4];
#pragma unroll
        for (int c = 0; c < 4; c++)   // min(127, round(t)) as i8: clamped first, NaN to 127; |t| is at most 128 and rounding then
            q[c] = (uint32_t)cq_round_away_i32(fmaxf(fminf(iscale * v[c], 127.0f), -128.0f));
        const uint32_t p01 = __builtin_amdgcn_perm(q[1], q[0], 0x0c0c0400u), p23 = __builtin_amdgcn_perm(q[3], q[2], 0x04000c0cu);
        packed[i] = any ? p01 | p23 : 0u;
        sum[i] = __builtin_amdgcn_sdot4((int)packed[i], 0x01010101, 0, false);
        sum[i] += dpp_i<kQuadSwap1>(sum[i]);
        sum[i] += dpp_i<kQuadSwap2>(sum[i]);   // bsums[4i + l / 4]
    }
    const int j = l & 3;
    bsum = j == 0 ? sum[0] : j == 1 ? sum[1] : j == 2 ? sum[2] : sum[3];
}

// The same for a block per wave: lane l holds elements 4l .. 4l + 3 in `f` and their quants in `packed`; `sum` is that of its four lanes (bsums[l / 4]),
// `d` the same in all.  For few blocks: the launch waits for one chain of dependent instructions, which the search for the first largest element,
// the rounding by itself and the clamp by another made twice as long.  Kernel alone, us: eight rows of 4096 3.00 -> 2.84, four behind rms_norm
// 4.84 -> 4.44, four of 14336 behind silu * mul 3.96 -> 3.96; in the calls that is 0.3 to 0.4 % (a step's 17 such launches among 41: 476.7 -> 474.6 us,
// eight rows with their matmul 10.21 -> 10.18).
__device__ __forceinline__ void cq_q8k_of_wave(const float4 f, int lane, uint32_t &packed, float &d, int &sum) {
    float hi = fmaxf(fmaxf(fmaxf(fmaxf(0.0f, f.x), f.y), f.z), f.w), lo = fminf(fminf(fminf(fminf(0.0f, f.x), f.y), f.z), f.w);
    hi = fmaxf(hi, dpp_f<kQuadSwap1>(hi));
    lo = fminf(lo, dpp_f<kQuadSwap1>(lo));
    hi = fmaxf(hi, dpp_f<kQuadSwap2>(hi));
    lo = fminf(lo, dpp_f<kQuadSwap2>(lo));
    hi = fmaxf(hi, dpp_f<kHalfMirror>(hi));
    lo = fminf(lo, dpp_f<kHalfMirror>(lo));
    hi = fmaxf(hi, dpp_f<kRowMirror>(hi));
    lo = fminf(lo, dpp_f<kRowMirror>(lo));
    hi = fmaxf(fmaxf(readlane_f(hi, 0), readlane_f(hi, 16)), fmaxf(readlane_f(hi, 32), readlane_f(hi, 48)));
    lo = fminf(fminf(readlane_f(lo, 0), readlane_f(lo, 16)), fminf(readlane_f(lo, 32), readlane_f(lo, 48)));
    const float amax = fmaxf(hi, -lo);
    float max = hi > -lo ? hi : lo;
    if (__any(hi == -lo && amax != 0.0f)) {   // both signs: the sign of the first of them
        int idx = 0x7fffffff;
        const float v[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
        for (int c = 3; c >= 0; c--)
            if (fabsf(v[c]) == amax) idx = 2 * (4 * lane + c) + (v[c] < 0.0f ? 1 : 0);
        max = wave_min_i(idx) & 1 ? lo : hi;
    }
    const bool any = amax != 0.0f;
    const float iscale = -128.0f / max;
    d = any ? 1.0f / iscale : 0.0f;
    const float v[4] = {f.x, f.y, f.z, f.w};
    uint32_t q[4];
#pragma unroll
    for (int c = 0; c < 4; c++) q[c] = (uint32_t)cq_round_away_i32(fmaxf(fminf(iscale * v[c], 127.0f), -128.0f));   // (as above)
    const uint32_t p01 = __builtin_amdgcn_perm(q[1], q[0], 0x0c0c0400u), p23 = __builtin_amdgcn_perm(q[3], q[2], 0x04000c0cu);
    packed = any ? p01 | p23 : 0u;
    sum = __builtin_amdgcn_sdot4((int)packed, 0x01010101, 0, false);
    sum += dpp_i<kQuadSwap1>(sum);
    sum += dpp_i<kQuadSwap2>(sum);
}

// Q8_0 / Q8_1 (k_quants.rs:586-615): a block per eight lanes, each with four consecutive elements `f` (zeros past the end of a row; called by
// all 64 lanes).  The four quants in a word, the unrounded scale, the block's sum.
__device__ __forceinline__ void cq_q8_0_of_eight(const float4 f, uint32_t &packed, float &d, int &sum) {
    float amax = fmaxf(fmaxf(fmaxf(fmaxf(0.0f, fabsf(f.x)), fabsf(f.y)), fabsf(f.z)), fabsf(f.w));
    amax = fmaxf(amax, dpp_f<kQuadSwap1>(amax));
    amax = fmaxf(amax, dpp_f<kQuadSwap2>(amax));
    amax = fmaxf(amax, dpp_f<kHalfMirror>(amax));  // quads hold one value each: the mirror pairs them
    d = amax / 127.0f;
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    const int8_t q0 = cq_as_i8(roundf(f.x * id)), q1 = cq_as_i8(roundf(f.y * id)), q2 = cq_as_i8(roundf(f.z * id)), q3 = cq_as_i8(roundf(f.w * id));
    sum = (int)q0 + (int)q1 + (int)q2 + (int)q3;
    sum += dpp_i<kQuadSwap1>(sum);
    sum += dpp_i<kQuadSwap2>(sum);
    sum += dpp_i<kHalfMirror>(sum);
    packed = (uint32_t)(uint8_t)q0 | ((uint32_t)(uint8_t)q1 << 8) | ((uint32_t)(uint8_t)q2 << 16) | ((uint32_t)(uint8_t)q3 << 24);
}
#endif
