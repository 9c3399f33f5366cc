// fno_dev.h -- device helpers shared by the FNO runtime's kernels
// (fno_rt.hip, fno_tail.hip): the reference Linear's step, the activations
// and fake-quants, the token tiles and the layer tail's element.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"
#include "fno_rt.h"
#include "gelu_exact.h"
#include "launch.h"
#include "snap.h"

namespace nfq {

__device__ __forceinline__ float rt_activate(float y, int act) {
    if (act == RT_ACT_RELU) return y < 0.0f ? 0.0f : y;  // fno.cpp:37-40
    if (act == RT_ACT_GELU) return gelu_fast<kGeluRefine>(y);
    return y;
}

// LDS written by some lanes of a wave, read by others after this point.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------
// fp32 Linear (fno.cpp:69-79) in the reference build's summation order: the
// first k - k % 8 products rounded and added one by one, the rest fused.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float lin_step(float acc, float x, float w, bool plain) {
    return plain ? acc + x * w : __builtin_fmaf(x, w, acc);
}

struct Tile {
    int64_t s;
    int t0, c0;
};

// Tile `id` of TT tokens x 64 channels.
template <int TT>
__device__ __forceinline__ bool tile_of(int64_t id, int64_t samples, int n, int w, Tile& tl) {
    const int tt = (n + TT - 1) / TT, tc = (w + 63) / 64;
    const int64_t per_sample = static_cast<int64_t>(tt) * tc;
    if (id >= samples * per_sample) return false;
    tl.s = id / per_sample;
    const int rem = static_cast<int>(id % per_sample);
    tl.t0 = (rem / tc) * TT;
    tl.c0 = (rem % tc) * 64;
    return true;
}

// fno.cpp:579-606 with the exponent e = int(std::round(log2|v| * 8) / 8)
// read off the step points of the reference's libm (thr: the smallest float
// of each exponent from -5 to 9, computed on the host with that libm):
// e = -6 + #{thr <= |v|} for 2^-6 <= |v| <= FLT_MAX, taken from |v|'s binade
// and one compare (snap.h; thr in LDS); NaN and Inf give ldexp(1, INT_MIN)
// = 0; 2^e for e >= 9 is capped at 448.
__device__ __forceinline__ float log2_snap(float x, float s, const float* thr) {
    const float v = x / s;
    const float av = fabsf(v);
    const float sign = v < 0.0f ? -1.0f : 1.0f;
    float qv;
    if (av < 0.015625f) {
        qv = av;
    } else if (!(av <= 0x1.fffffep+127f)) {
        qv = 0.0f;
    } else {
        const int e = snap_exponent_binade(av, thr);
        qv = e >= 9 ? 448.0f : __builtin_bit_cast(float, static_cast<uint32_t>(127 + e) << 23);
    }
    const float clamped = (448.0f < qv) ? 448.0f : qv;
    return (sign * clamped) * s;
}

// x2_fake_quant with the per-tensor scale's reciprocal inv = fl(1 / s)
// computed once (inv_ok: inv a normal float).  t = v * inv is within
// 1.5 * 2^-23 |t| of the quotient fl(v / s), so while |t| is farther than
// 2^-20 |t| from the nearest half-integer, rint(t) equals round(fl(v / s))
// (the two rounding rules differ only on ties) and the rest of the
// fake-quant follows unchanged; otherwise (near a tie, |t| >= 2^22, NaN,
// Inf) the exact division.
__device__ __forceinline__ float x2_fake_quant_inv(float v, float s, float inv, bool inv_ok, float zpf) {
    const float t = v * inv;
    const float at = fabsf(t);
    const float dist = fabsf(__builtin_amdgcn_fractf(at) - 0.5f);
    if (!(inv_ok && dist > __builtin_fmaf(at, 0x1p-20f, 0x1p-40f))) return x2_fake_quant(v, s, zpf);
    float q = rintf(t) + zpf;
    q = q < -128.0f ? -128.0f : q;
    q = q > 127.0f ? 127.0f : q;
    return (q - zpf) * s;
}

// The reciprocal of a per-tensor scale and whether it is a normal float.
struct ScaleInv {
    float inv;
    bool ok;
};
__device__ __forceinline__ ScaleInv scale_inv(float s) {
    const float inv = 1.0f / s;
    const float a = fabsf(inv);
    return {inv, a >= 0x1p-126f && a <= 0x1.fffffep+127f};
}

// Copies a step table into LDS; every thread of the block must call it.
__device__ __forceinline__ void stage_steps(float* steps, const float* thr) {
    if (threadIdx.x < 15) steps[threadIdx.x] = thr[threadIdx.x];
    __syncthreads();
}

// One element of the layer tail (fno.cpp:572-660): the x2 fake-quant KIND (0
// none, 1 per tensor, 2 per position, 3 log2 snap), act(x1 + x2), the next
// layer's input fake-quant FQN (0 off, 1 per tensor, 3 log2 snap).
template <int KIND, int ACT, int FQN>
__device__ __forceinline__ float post_element(float x1, float x2, const PostArgs& a, const ScaleInv& inv_x2,
                                              const ScaleInv& inv_next, const float* thr_x2,
                                              const float* thr_next, float pscale, float pzp) {
    if constexpr (KIND == 1) x2 = x2_fake_quant_inv(x2, a.scale, inv_x2.inv, inv_x2.ok, a.zpf);
    else if constexpr (KIND == 2) x2 = x2_fake_quant(x2, pscale, pzp);
    else if constexpr (KIND == 3) x2 = log2_snap(x2, a.scale, thr_x2);
    float y = x1 + x2;
    if constexpr (ACT == RT_ACT_RELU) y = y < 0.0f ? 0.0f : y;   // fno.cpp:37-40
    else if constexpr (ACT == RT_ACT_GELU) y = gelu_fast<kGeluRefine>(y);
    if constexpr (FQN == 1) y = x2_fake_quant_inv(y, a.fq_next.scale, inv_next.inv, inv_next.ok, a.fq_next.zpf);
    else if constexpr (FQN == 3) y = log2_snap(y, a.fq_next.scale, thr_next);
    return y;
}

// Tiles of tt tokens x 64 channels of a launch.
inline int64_t tile_count(int64_t samples, int n, int w, int tt) {
    return samples * ((n + tt - 1) / tt) * static_cast<int64_t>((w + 63) / 64);
}

}  // namespace nfq
