// nflow_quant.hip -- kernels and extern "C" entry points of libnflow_quant
// (declared in include/nflow_quant.h).
//
// Dispatch: the row-tile MFMA kernel (rows_kernel.h) serves every shape with
// K % 4 == 0, K <= 256 (fp32 input) or K <= 1024 (code input), N % 4 == 0
// and aligned pointers; anything else goes through the generic path
// (quantise kernel into a stream-ordered workspace, then one thread per
// output).  Both paths produce identical bits.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <utility>

#include "nflow_quant.h"
#include "common.h"
#include "launch.h"
#include "rows_kernel.h"
#include "chain_kernel.h"
#include "status.h"

namespace nfq {

// ---------------------------------------------------------------------------
// Elementwise / per-row kernels
// ---------------------------------------------------------------------------

// The elementwise kernels are bound by HBM.  A thread takes kElemQuads groups
// of four elements, 256 groups apart: 16-byte and 4-byte accesses of whole
// wave-contiguous segments, all of a thread's loads in flight at once; one
// group (per = 1) where four would leave the CUs under two blocks; the last
// n % 4 elements, and buffers the accesses do not fit (per = 0), go one by one,
// an element per thread.  (That form alone ran E4M3 encode 23.0 and decode
// 18.6 us at 16 Mi elements, 84 MB each; this one 16.4 and 12.8.  With the
// four-group grid throughout, decode of 1 Mi ran 3.6 us for 3.3, and an
// unaligned encode of 1 Mi 6.3.)
constexpr int kElemQuads = 4;

// f4(first quad, end of the block's quads) over whole quads, f1(element index)
// over the rest.
template <typename F4, typename F1>
__device__ __forceinline__ void each_quad(int64_t n, int per, F4 f4, F1 f1) {
    const int64_t nq = per ? n / 4 : 0, span = 256 * per;
    for (int64_t b = static_cast<int64_t>(blockIdx.x) * span; b < nq; b += static_cast<int64_t>(gridDim.x) * span)
        f4(b + threadIdx.x, b + span < nq ? b + span : nq);
    for (int64_t i = 4 * nq + static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * 256)
        f1(i);
}

// The launch of an elementwise kernel over n elements: groups per thread, grid.
static int elem_per(int64_t n, bool aligned_buffers) {
    return !aligned_buffers ? 0 : n / 4 <= static_cast<int64_t>(num_cus()) * 2 * 256 * kElemQuads ? 1 : kElemQuads;
}
static dim3 elem_grid(int64_t n, int per) {
    return dim3(per ? grid_for((n + 3) / 4, 256 * per, 16) : grid_for(n, 256, 16));
}

// QuantiseActivation, int8_gemm.cpp:507-520.
__global__ __launch_bounds__(256) void k_quantise_fixed(const float* __restrict__ A,
                                                        int8_t* __restrict__ Aq, int64_t n,
                                                        float s, int32_t zp, int per) {
    const float inv = 1.0f / s;
    const bool fast = s >= 0x1p-120f && s <= 0x1p120f;   // the reciprocal path's range
    each_quad(
        n, per,
        [&](int64_t q0, int64_t nq) {
            v4f x[kElemQuads];
#pragma unroll
            for (int u = 0; u < kElemQuads; ++u)
                if (q0 + 256 * u < nq) x[u] = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(A) + q0 + 256 * u);
#pragma unroll
            for (int u = 0; u < kElemQuads; ++u) {
                if (q0 + 256 * u >= nq) continue;
                reinterpret_cast<uint32_t*>(Aq)[q0 + 256 * u] = quant_i8_fixed4(x[u], s, inv, zp, fast);
            }
        },
        [&](int64_t i) { Aq[i] = static_cast<int8_t>(quant_i8_exact(A[i], s, zp)); });
}

// One wave per row: absmax -> scale -> codes (+ sum of codes).
// Weight-row byte sums the tiled GEMM's row-VNNI term needs next to a
// caller's sum_W (int8_gemm.cpp:386-393), formed by the quantise launch that
// runs just before the GEMM instead of a launch of their own.  out == null:
// none wanted.
struct CodeSums {
    const uint8_t* W;   // (N, K) int8 codes, 16-byte aligned rows
    int N;
    int K;              // a multiple of 16
    int32_t* out;       // (N)
};

// Rows 4 wg .. 4 wg + 3 of cs.W: 16 lanes per row, DPP row reductions.
__device__ __forceinline__ void code_sums_group(const CodeSums& cs, int64_t wg) {
    const int lane = threadIdx.x & 63, c = lane & 15;
    const int64_t n = wg * 4 + (lane >> 4);
    int32_t acc = 0;
    if (n < cs.N) {
        const v4u* w = reinterpret_cast<const v4u*>(cs.W + n * cs.K);
        for (int j = c; j < cs.K / 16; j += 16) {
            const v4u v = w[j];
#pragma unroll
            for (int q = 0; q < 4; ++q) acc = sum_bytes_i8(v[q], acc);
        }
    }
    acc += dpp_movi<0xB1>(acc);   // quad_perm [1,0,3,2]
    acc += dpp_movi<0x4E>(acc);   // quad_perm [2,3,0,1]
    acc += dpp_movi<0x141>(acc);  // row_half_mirror
    acc += dpp_movi<0x140>(acc);  // row_mirror
    if (c == 0 && n < cs.N) cs.out[n] = acc;
}

// Every wave of a quantise launch first takes its share of the weight rows.
__device__ __forceinline__ void code_sums_share(const CodeSums& cs) {
    if (!cs.out) return;
    const int64_t nw = static_cast<int64_t>(gridDim.x) * 4;
    for (int64_t wg = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6); wg * 4 < cs.N; wg += nw)
        code_sums_group(cs, wg);
}

// Codes of (M, K) rows with one scale (K a multiple of 4, 16-byte aligned
// rows) and their row sums, for the tiled GEMM: a wave per row, four float4
// per lane in flight.  Bound by HBM.
__global__ __launch_bounds__(256) void k_quantise_fixed_rows(const float* __restrict__ A, int64_t M, int K,
                                                             uint8_t* __restrict__ Aq, float* __restrict__ scale,
                                                             int32_t* __restrict__ sum_a, float s, int32_t zp,
                                                             CodeSums cs) {
    code_sums_share(cs);
    const int lane = threadIdx.x & 63, kq = K / 4;
    const float inv = 1.0f / s;
    const bool fast = s >= 0x1p-120f && s <= 0x1p120f;   // the reciprocal path's range
    const int64_t nw = static_cast<int64_t>(gridDim.x) * 4;
    for (int64_t m = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6); m < M; m += nw) {
        const v4f* x4 = reinterpret_cast<const v4f*>(A + m * K);
        uint32_t* q4 = reinterpret_cast<uint32_t*>(Aq + m * K);
        int32_t sa = 0;
        for (int j = lane; j < kq; j += 256) {
            v4f x[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) x[u] = __builtin_nontemporal_load(x4 + (j + 64 * u < kq ? j + 64 * u : j));
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (j + 64 * u >= kq) continue;
                const uint32_t v = quant_i8_fixed4(x[u], s, inv, zp, fast);
                q4[j + 64 * u] = v;
                sa = sum_bytes_i8(v, sa);
            }
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) sa += __shfl_xor(sa, o);
        if (lane == 0) {
            sum_a[m] = sa;
            scale[m] = s;      // the persistent GEMM reads its rows' scales
        }
    }
}

template <bool FP8>
__global__ __launch_bounds__(256) void k_quantise_token(const float* __restrict__ A, int64_t M,
                                                        int K, uint8_t* __restrict__ Aq,
                                                        float* __restrict__ scale,
                                                        int32_t* __restrict__ sum_a,
                                                        CodeSums cs) {
    code_sums_share(cs);
    const int lane = threadIdx.x & 63;
    const int64_t nw = static_cast<int64_t>(gridDim.x) * 4;
    for (int64_t m = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6); m < M; m += nw) {
        const float* x = A + m * K;
        float mx = 0.0f;
        for (int k = lane; k < K; k += 64) mx = fmaxf(mx, fabsf(x[k]));
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
        const float s = (mx == 0.0f) ? 1.0f : mx / (FP8 ? 448.0f : 127.0f);
        int32_t sa = 0;
        if constexpr (FP8) {
            const float inv = (s == 0.0f) ? 1.0f : 1.0f / s;
            for (int k = lane; k < K; k += 64) Aq[m * K + k] = static_cast<uint8_t>(fp8_quant(x[k], inv));
        } else {
            const float inv = 1.0f / s;
            for (int k = lane; k < K; k += 64) {
                const int32_t q = quant_i8_token(x[k], s, inv);
                Aq[m * K + k] = static_cast<uint8_t>(q);
                sa += q;
            }
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) sa += __shfl_xor(sa, o);
        }
        if (lane == 0) {
            scale[m] = s;
            if (sum_a) sum_a[m] = sa;
        }
    }
}

// PrecomputeSumW, int8_gemm.cpp:479-496: one wave per output row.
__global__ __launch_bounds__(256) void k_sum_w(const int8_t* __restrict__ W,
                                               const int32_t* __restrict__ zp, int K, int N,
                                               int32_t* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    const int o = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (o >= N) return;
    uint32_t acc = 0;
    for (int i = lane; i < K; i += 64)
        acc += static_cast<uint32_t>(static_cast<int32_t>(W[static_cast<int64_t>(o) * K + i]) - zp[o]);
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) acc += __shfl_xor(acc, s);
    if (lane == 0) out[o] = static_cast<int32_t>(acc);
}

// The weight-row byte sums on their own (linear_forward_quantised, which has
// no quantise launch to carry them).
__global__ __launch_bounds__(256) void k_code_sums(CodeSums cs) { code_sums_share(cs); }

// The bytes e4m3_encode(x[e]): the hardware conversion up to 448 in magnitude
// (where it and fp8_quant's clamp agree), else the encoder itself (448 to 464
// rounds down, (464, 496) is the NaN byte, larger is 448).
__device__ __forceinline__ uint32_t e4m3_encode4(v4f x) {
    const float m = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3])));
    if (m > 448.0f)
        return e4m3_encode(x[0]) | (e4m3_encode(x[1]) << 8) | (e4m3_encode(x[2]) << 16) | (e4m3_encode(x[3]) << 24);
    return fp8_pack4(x, 1.0f);
}

__global__ __launch_bounds__(256) void k_e4m3_encode(const float* __restrict__ in,
                                                     uint8_t* __restrict__ out, int64_t n, int per) {
    each_quad(
        n, per,
        [&](int64_t q0, int64_t nq) {
            v4f x[kElemQuads];
#pragma unroll
            for (int u = 0; u < kElemQuads; ++u)
                if (q0 + 256 * u < nq) x[u] = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(in) + q0 + 256 * u);
#pragma unroll
            for (int u = 0; u < kElemQuads; ++u)
                if (q0 + 256 * u < nq) reinterpret_cast<uint32_t*>(out)[q0 + 256 * u] = e4m3_encode4(x[u]);
        },
        [&](int64_t i) { out[i] = static_cast<uint8_t>(e4m3_encode(in[i])); });
}

__global__ __launch_bounds__(256) void k_e4m3_decode(const uint8_t* __restrict__ in,
                                                     float* __restrict__ out, int64_t n, int per) {
    each_quad(
        n, per,
        [&](int64_t q0, int64_t nq) {
            uint32_t b[kElemQuads];
#pragma unroll
            for (int u = 0; u < kElemQuads; ++u)
                if (q0 + 256 * u < nq) b[u] = reinterpret_cast<const uint32_t*>(in)[q0 + 256 * u];
#pragma unroll
            for (int u = 0; u < kElemQuads; ++u) {
                if (q0 + 256 * u >= nq) continue;
                v4f y;
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] = e4m3_decode((b[u] >> (8 * e)) & 0xFFu);
                __builtin_nontemporal_store(y, reinterpret_cast<v4f*>(out) + q0 + 256 * u);
            }
        },
        [&](int64_t i) { out[i] = e4m3_decode(in[i]); });
}

// fp8_e4m3_per_tensor_fake_quant, fp8_e4m3.h:312-334 (in == out allowed).
__global__ __launch_bounds__(256) void k_fp8_fake_quant(const float* in, float scale, float* out,
                                                        int64_t n, int per) {
    const float inv = (scale == 0.0f) ? 1.0f : (1.0f / scale);
    // The byte's value; the byte of a NaN decodes to the positive quiet NaN.
    auto value = [&](float x) {
        const float xs = x * inv;
        return (__builtin_isnan(xs) ? __uint_as_float(0x7FC00000u) : fp8_value_of(xs)) * scale;
    };
    each_quad(
        n, per,
        [&](int64_t q0, int64_t nq) {
            v4f x[kElemQuads];
#pragma unroll
            for (int u = 0; u < kElemQuads; ++u)
                if (q0 + 256 * u < nq) x[u] = reinterpret_cast<const v4f*>(in)[q0 + 256 * u];
#pragma unroll
            for (int u = 0; u < kElemQuads; ++u) {
                if (q0 + 256 * u >= nq) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e) x[u][e] = value(x[u][e]);
                reinterpret_cast<v4f*>(out)[q0 + 256 * u] = x[u];
            }
        },
        [&](int64_t i) { out[i] = value(in[i]); });
}

// Generic product + epilogue: one thread per output, any K / N / alignment.
// Codes are read from Aq (already quantised); per-row scale from scale_in
// (or the fixed a.scale_A when scale_in is null).
template <bool FP8, int OUT>
__global__ __launch_bounds__(256) void k_generic(RowsArgs a, int act) {
    const int64_t total = a.M * a.N;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
    const int K = a.K;
    const int Kd = std::min(K, a.kb_dot * 64);
    for (int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; idx < total;
         idx += stride) {
        const int64_t m = idx / a.N;
        const int n = static_cast<int>(idx - m * a.N);
        const uint8_t* x = a.Aq + m * K;
        const uint8_t* w = a.W + static_cast<int64_t>(n) * K;
        if constexpr (FP8) {
            float acc = 0.0f;
            for (int k = 0; k < Kd; ++k) acc += e4m3_decode(x[k]) * e4m3_decode(w[k]);
            if constexpr (OUT == OUT_RAW) {
                static_cast<float*>(a.C)[idx] = acc;
            } else {
                const float sa = a.scale_in ? a.scale_in[m] : a.scale_A;
                const float b = a.bias ? a.bias[n] : 0.0f;
                static_cast<float*>(a.C)[idx] = activate_rt(dequant_bias(a.sW[n], sa, acc, b), act);
            }
        } else {
            uint32_t D = 0, SA = 0, Sf = 0, Sd = 0;
            for (int k = 0; k < K; ++k) {
                const int32_t xv = static_cast<int8_t>(x[k]);
                const int32_t wv = static_cast<int8_t>(w[k]);
                SA += static_cast<uint32_t>(xv);
                Sf += static_cast<uint32_t>(wv);
                if (k < Kd) {
                    D += static_cast<uint32_t>(xv * wv);
                    Sd += static_cast<uint32_t>(wv);
                }
            }
            if constexpr (OUT == OUT_RAW) {
                static_cast<int32_t*>(a.C)[idx] = static_cast<int32_t>(D);
            } else {
                const int32_t zpw = a.zpW ? a.zpW[n] : 0;
                const int32_t swg = a.sumW ? a.sumW[n] : 0;
                const IntEpi e = int_epi_consts(a.formula, K, a.zp_A, zpw, swg, a.sumW != nullptr,
                                                static_cast<int32_t>(Sf), static_cast<int32_t>(Sd));
                // Not int_epi_value: its two-way sum spoils the compiler's
                // loop above (3089 x 1028 -> 156 659 -> 986 us).
                const int32_t t32 = int_epi_t32(e, static_cast<int32_t>(D), static_cast<int32_t>(SA));
                const float t = e.c2 == 0 ? static_cast<float>(t32) : static_cast<float>(static_cast<int64_t>(t32) + e.c2);
                const float sa = a.scale_in ? a.scale_in[m] : a.scale_A;
                const float b = a.bias ? a.bias[n] : 0.0f;
                static_cast<float*>(a.C)[idx] = activate_rt(dequant_bias(a.sW[n], sa, t, b), act);
            }
        }
    }
}

// Code stores are written through the L2 (sc1): the codes then need no
// write-back at the end of the launch before the product reads them
// (measured on the 65536-row 1024-wide layer: 128.5-129.9 -> 125.3 us per
// layer; nt 144 us, the product then reading them from HBM).
constexpr int kCodeCpol = 16;

// The same for rows of K = 256 KV floats: the row stays in registers (KV
// float4 per lane), so HBM is read once, in 1 KB wave instructions, and the
// codes leave as one dword per lane per float4.
template <bool FP8, int KV>
__global__ __launch_bounds__(256) void k_quantise_rows(const float* __restrict__ A, int64_t M,
                                                       uint8_t* __restrict__ Aq,
                                                       float* __restrict__ scale,
                                                       int32_t* __restrict__ sum_a,
                                                       CodeSums cs) {
    code_sums_share(cs);
    constexpr int K = 256 * KV;
    const int lane = threadIdx.x & 63;
    const int64_t nw = static_cast<int64_t>(gridDim.x) * 4;
    for (int64_t m = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6); m < M; m += nw) {
        const v4f* x4 = reinterpret_cast<const v4f*>(A + m * K);
        v4f x[KV];
#pragma unroll
        for (int i = 0; i < KV; ++i) x[i] = __builtin_nontemporal_load(x4 + lane + 64 * i);
        float mx = 0.0f;
#pragma unroll
        for (int i = 0; i < KV; ++i)
            mx = fmaxf(fmaxf(mx, fmaxf(fabsf(x[i][0]), fabsf(x[i][1]))), fmaxf(fabsf(x[i][2]), fabsf(x[i][3])));
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
        const float s = (mx == 0.0f) ? 1.0f : mx / (FP8 ? 448.0f : 127.0f);
        const auto qr = __builtin_amdgcn_make_buffer_rsrc(Aq + m * K, 0, K, 0x00020000);
        int32_t sa = 0;
        if constexpr (FP8) {
            const float inv = (s == 0.0f) ? 1.0f : 1.0f / s;
#pragma unroll
            for (int i = 0; i < KV; ++i)
                __builtin_amdgcn_raw_buffer_store_b32(fp8_pack4(x[i], inv), qr, 4 * (lane + 64 * i), 0, kCodeCpol);
        } else {
            const float inv = 1.0f / s;
#pragma unroll
            for (int i = 0; i < KV; ++i) {
                const uint32_t w = pack4(quant_i8_token(x[i][0], s, inv), quant_i8_token(x[i][1], s, inv),
                                         quant_i8_token(x[i][2], s, inv), quant_i8_token(x[i][3], s, inv));
                __builtin_amdgcn_raw_buffer_store_b32(w, qr, 4 * (lane + 64 * i), 0, kCodeCpol);
                sa = sum_bytes_i8(w, sa);
            }
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) sa += __shfl_xor(sa, o);
        }
        if (lane == 0) {
            scale[m] = s;
            if (sum_a) sum_a[m] = sa;
        }
    }
}

// Rows of K = 256 KV floats with KV <= 2: 16 lanes per row, so a wave holds
// four rows and every reduction is four DPP row steps.  The 64-lane form
// above waits on six cross-lane shuffles per reduction, which holds it to
// about 60% of a streaming copy at K = 256; this form reaches 88%.
// Lane (r, c) = (lane / 16, lane % 16) holds the float4s c + 16 j, j < 4 KV,
// of row 4 w + r: each load instruction reads 256 contiguous bytes of each
// of the four rows, and each code store writes 64.
template <bool FP8, int KV>
__global__ __launch_bounds__(256) void k_quantise_rows16(const float* __restrict__ A, int64_t M,
                                                         uint8_t* __restrict__ Aq,
                                                         float* __restrict__ scale,
                                                         int32_t* __restrict__ sum_a,
                                                         CodeSums cs) {
    code_sums_share(cs);
    constexpr int K = 256 * KV, J = 4 * KV;
    const int lane = threadIdx.x & 63, c = lane & 15;
    const int64_t nw = static_cast<int64_t>(gridDim.x) * 4;
    for (int64_t w = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6); w * 4 < M; w += nw) {
        const int64_t m = w * 4 + (lane >> 4);
        const bool live = m < M;
        const v4f* x4 = reinterpret_cast<const v4f*>(A + (live ? m : M - 1) * K);
        v4f x[J];
#pragma unroll
        for (int j = 0; j < J; ++j) x[j] = __builtin_nontemporal_load(x4 + c + 16 * j);
        float mx = 0.0f;
#pragma unroll
        for (int j = 0; j < J; ++j)
            mx = fmaxf(fmaxf(mx, fmaxf(fabsf(x[j][0]), fabsf(x[j][1]))), fmaxf(fabsf(x[j][2]), fabsf(x[j][3])));
        mx = fmaxf(mx, dpp_mov<0xB1>(mx));   // quad_perm [1,0,3,2]
        mx = fmaxf(mx, dpp_mov<0x4E>(mx));   // quad_perm [2,3,0,1]
        mx = fmaxf(mx, dpp_mov<0x141>(mx));  // row_half_mirror
        mx = fmaxf(mx, dpp_mov<0x140>(mx));  // row_mirror
        const float s = (mx == 0.0f) ? 1.0f : mx / (FP8 ? 448.0f : 127.0f);
        // The wave's four rows as one buffer range clipped at M (rows past
        // it are dropped by the hardware).
        const int64_t left = M - w * 4 < 4 ? M - w * 4 : 4;
        const auto qr = __builtin_amdgcn_make_buffer_rsrc(Aq + w * 4 * K, 0, static_cast<int>(left * K), 0x00020000);
        const int qoff = (lane >> 4) * K;
        int32_t sa = 0;
        if constexpr (FP8) {
            const float inv = (s == 0.0f) ? 1.0f : 1.0f / s;
#pragma unroll
            for (int j = 0; j < J; ++j)
                __builtin_amdgcn_raw_buffer_store_b32(fp8_pack4(x[j], inv), qr, qoff + 4 * (c + 16 * j), 0, kCodeCpol);
        } else {
            const float inv = 1.0f / s;
#pragma unroll
            for (int j = 0; j < J; ++j) {
                uint32_t v = pack4(quant_i8_token(x[j][0], s, inv), quant_i8_token(x[j][1], s, inv),
                                   quant_i8_token(x[j][2], s, inv), quant_i8_token(x[j][3], s, inv));
                v = live ? v : 0u;
                __builtin_amdgcn_raw_buffer_store_b32(v, qr, qoff + 4 * (c + 16 * j), 0, kCodeCpol);
                sa = sum_bytes_i8(v, sa);
            }
            sa += dpp_movi<0xB1>(sa);
            sa += dpp_movi<0x4E>(sa);
            sa += dpp_movi<0x141>(sa);
            sa += dpp_movi<0x140>(sa);
        }
        if (c == 0 && live) {
            scale[m] = s;
            if (sum_a) sum_a[m] = sa;
        }
    }
}

// The FNO layer's tail for the kernels that do not fuse it: C holds x2
// (bias included); C = act(R + fq(x2)) with the optional x2 fake-quant of
// a.xq_* (fno.cpp:572-654) and R (the spectral branch x1) optional.  One
// block per row at a time, columns across the threads.
__global__ __launch_bounds__(256) void k_fno_post(float* __restrict__ C, const float* __restrict__ R,
                                                  RowsArgs a, int act) {
    const int N = a.N;
    for (int64_t m = blockIdx.x; m < a.M; m += gridDim.x) {
        const int pos = a.xq_kind == 2 ? static_cast<int>(m % a.xq_points) : 0;
        for (int j = threadIdx.x; j < N; j += blockDim.x) {
            const int64_t i = m * N + j;
            float x2 = C[i];
            if (a.xq_kind == 1) {
                x2 = x2_fake_quant(x2, a.xq_scale, a.xq_zpf);
            } else if (a.xq_kind == 2) {
                const int64_t idx = static_cast<int64_t>(j) * a.xq_points + pos;
                x2 = x2_fake_quant(x2, a.xq_scales[idx], static_cast<float>(a.xq_zps[idx]));
            }
            C[i] = activate_rt(R ? R[i] + x2 : x2, act);
        }
    }
}

// ---------------------------------------------------------------------------
// Launch helpers
// ---------------------------------------------------------------------------

template <bool FP8, int OUT>
static void launch_generic(const RowsArgs& a, int act, hipStream_t st) {
    const unsigned grid = grid_for(a.M * a.N, 256, 16);
    hipLaunchKernelGGL((k_generic<FP8, OUT>), dim3(grid), dim3(256), 0, st, a, act);
}

// Per-token quantise of (M, K) rows: the register-resident kernel for
// K = 256, 512, 1024, 2048, 4096 (16-byte aligned rows), else one wave per
// row with a loop over K.
template <bool FP8>
static void launch_quantise_token(const float* A, int64_t M, int K, uint8_t* Aq, float* scale,
                                  int32_t* sum_a, hipStream_t st,
                                  CodeSums cs = CodeSums{nullptr, 0, 0, nullptr}) {
    const dim3 grid(grid_for(M, 4, 16)), block(256);
    if (aligned(A, 16) && aligned(Aq, 4)) {
        // K <= 512: 16 lanes per row, a block takes 16 rows, 4 blocks per CU.
        // K >= 1024 keeps a row per wave: there the shuffles are a small share
        // of the row's time, and the 16-lane form has four times fewer waves
        // (measured on MI355X at M = 65536, K = 1024: 68 us against 64 us).
        const dim3 grid16(grid_for(M, 16, 4));
        switch (K) {
            case 256: hipLaunchKernelGGL((k_quantise_rows16<FP8, 1>), grid16, block, 0, st, A, M, Aq, scale, sum_a, cs); return;
            case 512: hipLaunchKernelGGL((k_quantise_rows16<FP8, 2>), grid16, block, 0, st, A, M, Aq, scale, sum_a, cs); return;
            case 1024: hipLaunchKernelGGL((k_quantise_rows<FP8, 4>), grid, block, 0, st, A, M, Aq, scale, sum_a, cs); return;
            case 2048: hipLaunchKernelGGL((k_quantise_rows<FP8, 8>), grid, block, 0, st, A, M, Aq, scale, sum_a, cs); return;
            case 4096: hipLaunchKernelGGL((k_quantise_rows<FP8, 16>), grid, block, 0, st, A, M, Aq, scale, sum_a, cs); return;
            default: break;
        }
    }
    hipLaunchKernelGGL((k_quantise_token<FP8>), grid, block, 0, st, A, M, K, Aq, scale, sum_a, cs);
}

static int env_int(const char* name) {
    const char* v = std::getenv(name);
    return (v && v[0]) ? std::atoi(v) : 0;
}

// Initialised from the environment on first use (a thread-safe static).
KernelPath& kernel_path() {
    static KernelPath* k = [] {
        auto* p = new KernelPath();
        p->no_gemm.store(env_int("NFLOW_NO_GEMM"));
        p->no_rows64.store(env_int("NFLOW_NO_ROWS64"));
        p->no_token_gemm.store(env_int("NFLOW_NO_TOKEN_GEMM"));
        p->gemm_reg.store(env_int("NFLOW_GEMM_REG"));
        p->gemm_tile.store(env_int("NFLOW_GEMM_TILE"));
        p->gemm_mfma.store(env_int("NFLOW_GEMM_MFMA"));
        p->no_wide.store(env_int("NFLOW_NO_WIDE"));
        p->no_rows64_queue.store(env_int("NFLOW_NO_ROWS64_QUEUE"));
        p->no_layer_tail.store(env_int("NFLOW_NO_LAYER_TAIL"));
        p->generic_fft.store(env_int("NFLOW_GENERIC_FFT"));
        return p;
    }();
    return *k;
}

static int check_launch(const char* what) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(NFLOW_INTERNAL, std::string(what) + ": " + hipGetErrorString(e));
    return NFLOW_OK;
}

// Workspace of one call (codes, scales and sums between a quantise launch
// and the product that reads them), used only by this call's launches on
// its stream.  Each (device, stream) pair keeps one buffer that grows to the
// largest request and is reused by the next call on that stream: calls on
// one stream run in order, so the previous call's kernels are done with it
// before the next call's start.  The pair's lock is held for the call's
// lifetime, so host threads sharing a stream cannot interleave their launches
// inside one call.  A larger request frees the old buffer in stream order and
// allocates anew.  (A stream-ordered allocation and free per call cost about
// 10 us of host time, more than a 4096-row 1024-wide layer takes on the GPU.)
// The per-thread default stream (one handle for many streams) and a stream
// under graph capture (whose allocations belong to the graph) keep the
// per-call allocation.  Buffers live until the process ends.
struct WsEntry {
    std::mutex mu;
    void* p = nullptr;
    size_t cap = 0;
};

// Slot 0 is a call's own workspace; slot 1 holds the fp32 activations
// between the layers of nflow_int8_mlp_forward_per_token, whose per-layer
// calls take slot 0 meanwhile.
static WsEntry* ws_entry(int dev, hipStream_t st, int slot) {
    static std::mutex map_mu;
    static std::map<std::pair<int, uintptr_t>, std::unique_ptr<WsEntry>>* map =
        new std::map<std::pair<int, uintptr_t>, std::unique_ptr<WsEntry>>();
    std::lock_guard<std::mutex> g(map_mu);
    auto& e = (*map)[{dev * 2 + slot, reinterpret_cast<uintptr_t>(st)}];
    if (!e) e.reset(new WsEntry);
    return e.get();
}

struct Scratch {
    void* p = nullptr;
    hipStream_t st = nullptr;
    hipError_t err = hipSuccess;
    bool owned = false;                    // per-call allocation (freed here)
    std::unique_lock<std::mutex> lock;
    Scratch(size_t bytes, hipStream_t s, int slot = 0) : st(s) {
        if (path_flag(kernel_path().no_workspace)) {
            err = hipErrorOutOfMemory;
            return;
        }
        bytes = std::max<size_t>(bytes, 256);
        int dev = 0;
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (s == hipStreamPerThread || hipStreamIsCapturing(s, &cap) != hipSuccess ||
            cap != hipStreamCaptureStatusNone || hipGetDevice(&dev) != hipSuccess) {
            err = hipMallocAsync(&p, bytes, s);
            owned = err == hipSuccess;
            return;
        }
        WsEntry* e = ws_entry(dev, s, slot);
        lock = std::unique_lock<std::mutex>(e->mu);
        if (bytes > e->cap) {
            if (e->p) (void)hipFreeAsync(e->p, s);
            e->p = nullptr;
            e->cap = 0;
            const size_t want = (bytes + (size_t(2) << 20) - 1) & ~((size_t(2) << 20) - 1);
            err = hipMallocAsync(&e->p, want, s);
            if (err != hipSuccess) {
                e->p = nullptr;
                return;
            }
            e->cap = want;
        }
        p = e->p;
    }
    ~Scratch() {
        if (owned && p) (void)hipFreeAsync(p, st);
    }
    Scratch(const Scratch&) = delete;
    Scratch& operator=(const Scratch&) = delete;
};

// Whether a graph capture is recording stream st.  A workspace would then be
// allocated inside the graph (a chain of layers recorded that way took an
// illegal memory access on its first replay), so layers the one-pass kernel
// can serve take it, also where the split form is the faster one.
static bool stream_capturing(hipStream_t st) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(st, &cap) == hipSuccess && cap != hipStreamCaptureStatusNone;
}

static int kb_dot_for(int formula, int K) {
    if (formula == F_ROW_VNNI) return K / 64;   // int8_gemm.cpp:366: vec_end = K - K % 64
    return (K + 63) / 64;
}

static int formula_row(int K) { return K <= 4096 ? F_ROW_VNNI : F_ROW_SCALAR; }

// The tiled GEMM serves INT8 code input with K a multiple of 64, K >= 128
// (NFLOW_NO_GEMM=1 selects the row-tile kernel instead, for A/B timing).
static bool use_gemm(const RowsArgs& a) { return gemm_ok(a) && !path_flag(kernel_path().no_gemm); }

// Where a layer on fp32 input takes the row-tile kernel (weights in registers
// or re-read per 16 rows, no barriers) rather than the one-pass kernel.
// Measured on MI355X (us, row-tile / one-pass):
//   K, N <= 64: 300000 x 64 -> 40 26.9 either way; it stays;
//   per-token INT8 of K < 64 into a few more columns, many rows: 200000 x 8 ->
//     132 42.6 / 61, x 48 -> 68 34.5 / 45, but x 32 -> 256 120 / 70 and
//     40000 x 4 -> 132 16.6 / 15.6;
//   two K blocks into few columns, many rows: FP8 into 16 and fewer 30000 x 100
//     -> 16 7.3 / 8.6, 60000 10.4 / 14.0, but -> 20 14.0 / 14.2; fixed scale 60000 x 100
//     -> 20 12.4 / 15.4, -> 40 16.5 / 17.0, x 128 -> 20 15.2 / 15.8; per-token INT8
//     60000 x 100 -> 20 10.6 / 17.5, 350000 -> 48 64 / 80, x 128 -> 20 12.1 / 15.4, but
//     100000 x 128 -> 32 24.7 / 23.8 and 30000 x 128 -> 20 8.4 / 8.1.
static bool use_rows(const RowsArgs& a, int in_mode, bool fp8) {
    if (!rows_ok(a, in_mode)) return false;
    if (a.N <= 64 && a.K <= 64) return true;
    if (path_flag(kernel_path().token_rows)) return false;   // forced tiles: one-pass
    if (a.K > 64 && fp8) return a.N <= 16 && a.M >= 24576;
    if (a.K > 64) return a.N <= (a.K == 128 ? 20 : in_mode == IN_F32_TOKEN ? 48 : 40) && a.M >= 49152;
    return in_mode == IN_F32_TOKEN && !fp8 && a.K < 64 && a.N <= 160 && a.M >= 65536;
}

// Whether a layer on fp32 input that use_rows does not claim takes the one-pass
// kernel (token_gemm_kernel.h) rather than the generic one.
static bool use_token_gemm(const RowsArgs& a) {
    return token_gemm_ok(a) && !path_flag(kernel_path().no_token_gemm);
}

// Whether a layer on fp32 input takes the few-row kernel (skinny_kernel.h):
// while its 16 x 16 output blocks, which each quantise their rows for
// themselves, are few.  Measured on MI355X (us, few-row / the kernel that
// runs otherwise): static 1 x 1024 -> 1024 5.2 / 12.6, INT8 64 x 1024 -> 1024
// (256 blocks) 7.1 / 11.1, 128 x (512 blocks) 12.2 / 11.3; K <= 256 (4 waves
// per block) 300 x 200 -> 512 (608 blocks) 5.1 / 7.1, 2000 x 256 -> 64 (500)
// 4.9 / 5.5, 1000 x 256 -> 256 (1008) 6.4 / 5.5; K <= 128, where the one-pass
// kernel's chain is short, 300 x 64 -> 128 (152) 4.0 / 3.7; K = 4096, 1 -> 2048
// (128) 13 / 19, 128 rows (1024) 67 / 21.
static bool use_skinny(const RowsArgs& a) {
    const int f = kernel_path().skinny.load(std::memory_order_relaxed);
    if (f == 2 || !skinny_ok(a) || in_place(a)) return false;   // its blocks share rows
    if (f == 1) return true;
    const int64_t blocks = ((a.M + 15) / 16) * ((static_cast<int64_t>(a.N) + 15) / 16);
    const int64_t cus = num_cus();
    if (a.K <= 128 || a.K > 2048) return blocks <= cus / 2;
    return blocks <= (a.K <= 256 ? 2 * cus : cus);
}

// Per-token INT8 shapes the tiled GEMM could also take (after a quantise
// launch): whether that split is the faster form.  The one-pass kernel reads
// all the weights once per row tile, the split form reads the activations
// once and the codes per column block.  Measured on MI355X (us, one-pass /
// split) over K = 192 .. 512, 22 row counts from 600 to 100000, 12 widths:
//   K <= 256: one-pass for whole shapes (20000 x 256 -> 512 17.9 / 20.4).  The
//     masked form loses to the GEMM at K = 256 (3000 -> 1000 15.4 / 10.8, 20000 ->
//     300 21.9 / 18.1, 80000 -> 800 92 / 75; not in one nearly full round of nearly
//     full chunks, 32768 -> 500 27.4 / 29.6), below that with few 64-row tiles per
//     CU (6000 x 192 -> 640 13.8 / 10.5, 3000 x 128 -> 2000 15.1 / 11.8; 12000 x 192
//     -> 768 17.1 / 19.7, 12000 x 128 -> 800 15.7 / 17.6) and where a second round
//     is half empty (40000 x 192 -> 1000 58 / 52, 40000 x 128 -> 800 47 / 40), and at
//     K = 128 from N = 1024 on (6000 -> 2000 19.5 / 16.7; 20000 -> 2000 42 / 45);
//   larger K at 16-row tiles: one-pass up to 2.5 (row tile, 128-column chunk)
//     pairs per CU (2000 x 384 -> 500 9.2 / 9.7, 3000 -> 1000 16.9 / 12.3), 3.5 with
//     part lines at K = 512 (2500 x 512 -> 500 12.3 / 13.7, 2000 -> 1000 15.2 /
//     14.1), and for narrow N
//     throughout (8192 x 320 -> 300 11.6 / 13.2);
//   at 64-row tiles two blocks per CU work through the tiles in rounds: split
//     with at most a tile per CU (12000 x 384 -> 1024 29 / 27) and where the last
//     round leaves a third of the slots idle (20000 x 384 -> 300 29.7 / 26.5, 40000
//     x 320 -> 1000 76 / 64), one-pass elsewhere (32768 x 384 -> 576 36.5 / 45,
//     65536 x 448 -> 1024 97 / 152);
//   K = 512, where the persistent GEMM runs: split from N = 1024 (65536 110 / 88)
//     and from N = 512 beyond one round (65536 x 512 -> 576 74 / 68; 32768 37.5 /
//     40), one-pass with wide rows of part lines (16384 -> 1000 37.6 / 48).
static bool split_faster(const RowsArgs& a) {
    if (a.K > 512) return true;
    const int64_t cus = num_cus(), tiles = (a.M + 63) / 64;
    const int64_t pairs = ((a.M + 15) / 16) * ((static_cast<int64_t>(a.N) + 127) / 128);
    const int64_t slots = 2 * cus, rounds = (tiles + slots - 1) / slots;
    const int64_t fill = 100 * tiles / (rounds * slots);   // per cent, of the rounds' slots
    const bool part_lines = a.N % 32 != 0;
    if (a.K <= 256) {
        if (token_whole(a)) return false;
        if (a.K == 256) {
            const int chunks = (a.N + 255) / 256;
            if (tiles > cus && tiles <= slots && fill >= 75 && a.N >= 192 * chunks) return false;
            return a.N > 192 && 2 * pairs > 7 * cus;
        }
        if (token_small_tiles(a) || a.N <= (a.K == 128 ? 767 : 256)) return false;
        if (a.K == 128 && a.N >= 1024) return true;
        // Eighths of a tile per CU.
        const int eighths = a.K == 128 || (a.N > 640 && a.N < 2048) ? 4 : a.N <= 640 ? 6 : 3;
        return 8 * tiles <= eighths * cus || (tiles > slots && fill < 65);
    }
    if (token_small_tiles(a))
        return a.N > (a.K == 512 && !part_lines ? 255 : 384) && 2 * pairs > (a.K == 512 && part_lines ? 7 : 5) * cus;
    if (tiles < cus) return true;
    if (a.K < 512) return a.N > 256 && (tiles == cus || fill < 68);
    if (part_lines) return a.N <= 384 && tiles > cus && tiles <= slots && fill < 65;
    if (a.N >= 1024 || (a.N >= 512 && tiles > slots)) return true;
    return a.N > 256 && tiles > cus && fill < 65;
}

// The same choice for FP8 (K >= 512).  Measured on MI355X (us, one-pass /
// split): 1000 x 1024 -> 1024 17 / 11, 4096 x 1024 -> 1024 40 / 21; at K = 512
// 1000 -> 1024 10.2 / 9.5, 16384 -> 256 14.3 / 20.9, 16384 -> 1024 30 / 34.7, but
// 20000 -> 2048 79 / 64.
static bool fp8_split_faster(const RowsArgs& a) {
    if (kernel_path().token_rows.load(std::memory_order_relaxed)) return false;   // forced tiles: one-pass
    return a.K > 512 || (a.N > 1024 && !token_small_tiles(a));
}

// The same choice for fixed-scale INT8: one-pass for K <= 256, else as per token.
// Measured on MI355X (us, one-pass / split): 2000 x 320 -> 1024 12.4 / 9.5, 8192 ->
// 512 15.9 / 13.9; K = 512, 32768 -> 512 33.1 / 40.1, 8192 -> 2048 41.6 / 30.2; K =
// 1024 300 -> 256 13.6 / 11.6, 16384 -> 1024 150 / 45; at worst, with one tile per CU,
// 16384 x 320 -> 1024 28.2 / 33.3.
static bool fixed_split_faster(const RowsArgs& a) {
    if (kernel_path().token_rows.load(std::memory_order_relaxed)) return false;   // forced tiles: one-pass
    return a.K > 256 && split_faster(a);
}

// Fixed-scale int8 path shared by LinearForward / rows / batched.
static int int8_fixed_path(const nflow_int8_linear_params* p, int64_t rows, const float* A, float* C,
                           int formula, hipStream_t st, const char* what) {
    RowsArgs a{};
    a.A = A;
    a.M = rows;
    a.K = p->in_features;
    a.N = p->out_features;
    a.W = reinterpret_cast<const uint8_t*>(p->W_int8);
    a.sW = p->scale_W;
    a.zpW = p->zp_W;
    a.bias = p->bias;
    a.sumW = p->sum_W_per_row;
    a.scale_A = p->scale_A;
    a.zp_A = p->zp_A;
    a.formula = formula;
    a.kb_dot = kb_dot_for(formula, a.K);
    a.C = C;
    if (use_skinny(a)) {
        launch_skinny_i8_fixed(a, st);
        return check_launch(what);
    }
    if (rows64_ok(a) && !path_flag(kernel_path().no_rows64)) {
        launch_rows64_fixed(a, st);
        return check_launch(what);
    }
    if (use_rows(a, IN_F32_FIXED, false)) {
        launch_rows<false, IN_F32_FIXED, OUT_EPI>(a, ACT_NONE, st);
        return check_launch(what);
    }
    RowsArgs g = a;
    g.Aq = nullptr;  // the codes go to the workspace, which is 256-byte aligned
    const bool wide = aligned(A, 16) && use_gemm(g);
    // A few dozen products per row, many rows, N off 4: a thread per output on
    // codes (150000 x 4 -> 5 9.6 us, one-pass 20.9; x 16 -> 3 13.4 / 20.7; at
    // x 16 -> 5 both 21).
    const bool tiny = static_cast<int64_t>(a.K) * a.N <= 48 && rows >= 32768;
    if (use_token_gemm(a) && !((tiny || (wide && fixed_split_faster(a))) && !stream_capturing(st))) {
        launch_token_i8_fixed(a, st);
        return check_launch(what);
    }
    if (wide) {
        // Quantise (with the row sums, and the weight-row sums where the
        // formula takes them), then the tiled GEMM.
        const bool want_colsum = gemm_needs_colsum(a);
        const size_t codes16 = ((static_cast<size_t>(rows) * a.K + 15) / 16) * 16;
        Scratch ws(codes16 + (2 * static_cast<size_t>(rows) + (want_colsum ? a.N : 0)) * sizeof(int32_t), st);
        if (ws.err != hipSuccess && use_token_gemm(a)) {
            (void)hipGetLastError();
            launch_token_i8_fixed(a, st);
            return check_launch(what);
        }
        if (ws.err != hipSuccess) return set_error(NFLOW_INTERNAL, std::string(what) + ": workspace allocation failed");
        uint8_t* q = static_cast<uint8_t*>(ws.p);
        float* sc = reinterpret_cast<float*>(q + codes16);
        int32_t* sums = reinterpret_cast<int32_t*>(sc + rows);
        int32_t* colsum = want_colsum ? sums + rows : nullptr;
        hipLaunchKernelGGL(k_quantise_fixed_rows, dim3(grid_for(rows, 4, 16)), dim3(256), 0, st, A, rows, a.K, q, sc,
                           sums, p->scale_A, p->zp_A, CodeSums{a.W, a.N, a.K, colsum});
        a.Aq = q;
        a.scale_in = sc;
        a.sum_in = sums;
        a.colsum_in = colsum;
        launch_gemm<OUT_EPI>(a, ACT_NONE, st);
        return check_launch(what);
    }
    Scratch ws(static_cast<size_t>(rows) * a.K, st);
    if (ws.err != hipSuccess && use_token_gemm(a)) {
        (void)hipGetLastError();
        launch_token_i8_fixed(a, st);
        return check_launch(what);
    }
    if (ws.err != hipSuccess) return set_error(NFLOW_INTERNAL, std::string(what) + ": workspace allocation failed");
    const int64_t n = rows * a.K;
    const int per = elem_per(n, aligned(A, 16));
    hipLaunchKernelGGL(k_quantise_fixed, elem_grid(n, per), dim3(256), 0, st, A, static_cast<int8_t*>(ws.p), n,
                       p->scale_A, p->zp_A, per);
    a.Aq = static_cast<const uint8_t*>(ws.p);
    a.scale_in = nullptr;
    launch_generic<false, OUT_EPI>(a, ACT_NONE, st);
    return check_launch(what);
}

static int check_params(const nflow_int8_linear_params* p, const char* what) {
    if (!p || !p->W_int8 || !p->scale_W || !p->zp_W)
        return set_error(NFLOW_INVALID_ARG, std::string(what) + ": null input/output");
    if (p->in_features <= 0 || p->out_features <= 0)
        return set_error(NFLOW_INVALID_ARG, std::string(what) + ": bad feature dims");
    return NFLOW_OK;
}

static bool valid_act(int act) { return act == ACT_NONE || act == ACT_RELU || act == ACT_GELU_TANH; }

}  // namespace nfq

using namespace nfq;

extern "C" {

int nflow_quant_abi_version(void) { return NFLOW_QUANT_ABI_VERSION; }

int nflow_debug_set_kernel_path(const char* name, int value, int* previous) {
    clear_error();
    if (!name) return set_error(NFLOW_INVALID_ARG, "debug_set_kernel_path: null name");
    KernelPath& k = kernel_path();
    const std::string n(name);
    std::atomic<int>* f = n == "no_gemm" ? &k.no_gemm
                        : n == "no_rows64" ? &k.no_rows64
                        : n == "no_token_gemm" ? &k.no_token_gemm
                        : n == "token_rows" ? &k.token_rows
                        : n == "skinny" ? &k.skinny
                        : n == "gemm_reg" ? &k.gemm_reg
                        : n == "gemm_tile" ? &k.gemm_tile
                        : n == "gemm_mfma" ? &k.gemm_mfma
                        : n == "no_wide" ? &k.no_wide
                        : n == "no_rows64_queue" ? &k.no_rows64_queue
                        : n == "no_layer_tail" ? &k.no_layer_tail
                        : n == "no_workspace" ? &k.no_workspace
                        : n == "generic_fft" ? &k.generic_fft : nullptr;
    if (!f) return set_error(NFLOW_INVALID_ARG, "debug_set_kernel_path: unknown name " + n);
    const int old = f->exchange(value, std::memory_order_relaxed);
    if (previous) *previous = old;
    return NFLOW_OK;
}

int nflow_int8_quantise_activation(const float* A, int8_t* A_q, int64_t bsz, int in_features,
                                   float scale_A, int32_t zp_A, void* stream) {
    clear_error();
    if (!A || !A_q) return NFLOW_OK;   // the reference returns silently (int8_gemm.cpp:511)
    const int64_t n = bsz * static_cast<int64_t>(in_features);
    if (n <= 0) return NFLOW_OK;
    const int per = elem_per(n, aligned(A, 16) && aligned(A_q, 4));
    hipLaunchKernelGGL(k_quantise_fixed, elem_grid(n, per), dim3(256), 0, as_stream(stream), A, A_q, n, scale_A, zp_A,
                       per);
    return check_launch("QuantiseActivation");
}

int nflow_int8_precompute_sum_w(const int8_t* W_int8, const int32_t* zp_W, int in_features,
                                int out_features, int32_t* sum_W_out, void* stream) {
    clear_error();
    if (!W_int8 || !zp_W || !sum_W_out || in_features <= 0 || out_features <= 0)
        return set_error(NFLOW_INVALID_ARG, "PrecomputeSumW: null input or bad dims");
    hipLaunchKernelGGL(k_sum_w, dim3((out_features + 3) / 4), dim3(256), 0, as_stream(stream),
                       W_int8, zp_W, in_features, out_features, sum_W_out);
    return check_launch("PrecomputeSumW");
}

int nflow_int8_linear_forward(const nflow_int8_linear_params* p, const float* A, float* C,
                              void* stream) {
    clear_error();
    if (!A || !C) return set_error(NFLOW_INVALID_ARG, "Int8Linear: null input/output");
    int rc = check_params(p, "Int8Linear");
    if (rc) return rc;
    return int8_fixed_path(p, 1, A, C, formula_row(p->in_features), as_stream(stream),
                           "Int8Linear");
}

int nflow_int8_linear_forward_rows(const nflow_int8_linear_params* p, int64_t rows,
                                   const float* A, float* C, void* stream) {
    clear_error();
    if (!A || !C) return set_error(NFLOW_INVALID_ARG, "Int8Linear: null input/output");
    int rc = check_params(p, "Int8Linear");
    if (rc) return rc;
    if (rows <= 0) return NFLOW_OK;
    return int8_fixed_path(p, rows, A, C, formula_row(p->in_features), as_stream(stream),
                           "Int8Linear");
}

int nflow_int8_linear_forward_batched(const nflow_int8_linear_params* p, int64_t bsz,
                                      const float* A, float* C, void* stream) {
    clear_error();
    if (bsz <= 0) return NFLOW_OK;
    if (!A || !C) return set_error(NFLOW_INVALID_ARG, "LinearForwardBatched: null A or C");
    int rc = check_params(p, "LinearForwardBatched");
    if (rc) return rc;
    return int8_fixed_path(p, bsz, A, C, F_BATCHED, as_stream(stream), "LinearForwardBatched");
}

int nflow_int8_quantise_per_token(const float* A, int64_t M, int K, int8_t* A_q, float* scale_A,
                                  int32_t* sum_a, void* stream) {
    clear_error();
    if (!A || !A_q || !scale_A) return set_error(NFLOW_INVALID_ARG, "quantise_per_token: null pointer");
    if (K <= 0) return set_error(NFLOW_INVALID_ARG, "quantise_per_token: K <= 0");
    if (M <= 0) return NFLOW_OK;
    launch_quantise_token<false>(A, M, K, reinterpret_cast<uint8_t*>(A_q), scale_A, sum_a, as_stream(stream));
    return check_launch("quantise_per_token");
}

}  // extern "C"

namespace nfq {

// Per-token INT8 layer; with a residual R (M x N) the result is the FNO layer
// form act(R + x2): fused in the K = N = 64 kernel, else x2 then one pass.
// The x2 fake-quant parameters into a (nflow_x2_quant, fno.cpp:572-648).
static int apply_x2q(RowsArgs& a, const nflow_x2_quant* xq, const char* what) {
    if (!xq || xq->kind == NFLOW_X2_NONE) return NFLOW_OK;
    const std::string w(what);
    if (xq->kind == NFLOW_X2_PER_TENSOR) {
        a.xq_kind = 1;
        a.xq_scale = xq->scale;
        a.xq_zpf = static_cast<float>(xq->zero_point);
        return NFLOW_OK;
    }
    if (xq->kind == NFLOW_X2_PER_POSITION) {
        if (!xq->scales || !xq->zero_points) return set_error(NFLOW_INVALID_ARG, w + ": null per-position qparams");
        if (xq->points <= 0) return set_error(NFLOW_INVALID_ARG, w + ": per-position qparams need points > 0");
        if (xq->width != a.N)
            return set_error(NFLOW_SHAPE_MISMATCH, w + ": per-position qparam width differs from out_features");
        if (xq->n_positions < static_cast<int64_t>(a.N) * xq->points)
            return set_error(NFLOW_SHAPE_MISMATCH, w + ": fewer per-position qparams than out_features * points");
        a.xq_kind = 2;
        a.xq_scales = xq->scales;
        a.xq_zps = xq->zero_points;
        a.xq_points = xq->points;
        return NFLOW_OK;
    }
    if (xq->kind == NFLOW_X2_FP8_LOG2)
        return set_error(NFLOW_UNSUPPORTED_OP, w + ": the log2 FP8 snap of x2 is not an E4M3 operation");
    return set_error(NFLOW_INVALID_ARG, w + ": unknown x2 fake-quant kind");
}

// Device scratch of nflow_int8_linear_forward_per_token_noalloc: the split
// path's codes, scales and byte sums (at most kNoAllocScratchBytes).  Each
// GPU the library runs on holds its own copy until the process ends; the
// name is a host-side stand-in, so host code uses only the device address
// hipGetSymbolAddress returns for the current device.  Nothing in it needs
// to start at zero: the quantise launch writes every byte the product reads.
constexpr size_t kNoAllocScratchBytes = NFLOW_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

// The current device's address of `scratch`, looked up on the first call
// that needs it on that device and kept per device, and that device's lock
// on it: a call holds the lock from the lookup until its product is
// launched, so host threads whose calls share one stream cannot interleave
// their quantise and product launches on the one array (launches on
// different streams still run concurrently on the device and race).
constexpr int kMaxDevices = 64;
static std::mutex noalloc_mu[kMaxDevices];

static int noalloc_scratch_address(void** out, std::unique_lock<std::mutex>* hold) {
    static std::mutex mu;
    static void* addr[kMaxDevices] = {};
    int dev = 0;
    const hipError_t ed = hipGetDevice(&dev);
    if (ed != hipSuccess) return set_error(NFLOW_INTERNAL, std::string("noalloc scratch: hipGetDevice: ") + hipGetErrorString(ed));
    if (dev < 0 || dev >= kMaxDevices) return set_error(NFLOW_INTERNAL, "noalloc scratch: device index out of range");
    *hold = std::unique_lock<std::mutex>(noalloc_mu[dev]);
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
        void* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return set_error(NFLOW_INTERNAL, std::string("noalloc scratch: hipGetSymbolAddress: ") + hipGetErrorString(e));
        addr[dev] = ptr;
    }
    *out = addr[dev];
    return NFLOW_OK;
}

// The no-allocation entry point's workspace: the library's static device
// scratch of `cap` bytes, its address looked up (once per device) only after
// the shape has been checked against `cap`.  Null: allocate on the stream.
struct FixedWs {
    size_t cap;
    const char* what;
};

// The split path's workspace: codes, then (with no scale_A_out) M scales, then
// M row code sums when zero points may be nonzero and N weight-row byte sums
// when the formula takes a caller's sum_W (both for the tiled GEMM only).
static size_t split_sums(const RowsArgs& a, bool wide) {
    const bool want_sums = wide && a.zpW;
    const bool want_colsum = wide && a.formula == F_ROW_VNNI && a.sumW;
    return (want_sums ? static_cast<size_t>(a.M) : 0) + (want_colsum ? a.N : 0);
}
static size_t noalloc_need(const RowsArgs& a, bool wide) {
    const size_t codes16 = ((static_cast<size_t>(a.M) * a.K + 15) / 16) * 16;
    return codes16 + (a.scale_out ? 0 : static_cast<size_t>(a.M) * sizeof(float)) +
           split_sums(a, wide) * sizeof(int32_t);
}
// Shapes the no-allocation entry point documents as never touching its
// scratch: K = 128, 256 and 512 with N a multiple of 64, and K <= 256 the tiled
// GEMM cannot take (K, N multiples of 4), both at aligned buffers.  Calls on
// them are independent of every other call, on any stream.
static bool noalloc_scratch_free(const RowsArgs& a, bool wide) {
    const bool narrow = !wide && a.K <= 256 && a.K % 4 == 0 && a.N % 4 == 0 && aligned(a.A, 16) &&
                        aligned(a.W, 4) && aligned(a.C, 16);
    return token_whole(a) || narrow;
}
// Shapes it documents as too large for its scratch: the others whose codes
// the split path would hold there, also where the one-pass kernel, which needs
// none, would run them.
static bool noalloc_refuses(const RowsArgs& a, bool wide, size_t cap) {
    return !noalloc_scratch_free(a, wide) && noalloc_need(a, wide) > cap;
}

static int int8_per_token(const nflow_int8_linear_params* p, int64_t M, const float* A,
                          const float* R, float* C, float* scale_A_out, int activation,
                          const nflow_x2_quant* xq, void* stream, const FixedWs* fixed = nullptr) {
    if (!A || !C || !p || !p->W_int8 || !p->scale_W)
        return set_error(NFLOW_INVALID_ARG, "linear_forward_per_token: null input/output");
    if (p->in_features <= 0 || p->out_features <= 0)
        return set_error(NFLOW_INVALID_ARG, "linear_forward_per_token: bad feature dims");
    if (!valid_act(activation))
        return set_error(NFLOW_INVALID_ARG, "linear_forward_per_token: unknown activation");
    if (R && R == C) return set_error(NFLOW_INVALID_ARG, "fno_layer: x1 and y must be distinct buffers");
    RowsArgs a{};
    a.N = p->out_features;
    if (int rc = apply_x2q(a, xq, "fno_layer")) return rc;
    if (M <= 0) return NFLOW_OK;
    hipStream_t st = as_stream(stream);
    a.A = A;
    a.M = M;
    a.K = p->in_features;
    a.W = reinterpret_cast<const uint8_t*>(p->W_int8);
    a.sW = p->scale_W;
    a.zpW = p->zp_W;
    a.bias = p->bias;
    a.sumW = p->sum_W_per_row;
    a.zp_A = 0;
    a.formula = formula_row(a.K);
    a.kb_dot = kb_dot_for(a.formula, a.K);
    a.C = C;
    a.scale_out = scale_A_out;
    if (rows64_ok(a) && (!R || aligned(R, 16)) && !path_flag(kernel_path().no_rows64)) {
        a.residual = R;
        launch_rows64<false>(a, activation, st);
        return check_launch("linear_forward_per_token");
    }
    const bool post = R || a.xq_kind;
    const int act_x2 = post ? static_cast<int>(ACT_NONE) : activation;
    auto finish = [&]() {
        if (post) hipLaunchKernelGGL(k_fno_post, dim3(grid_for(M, 1, 16)), dim3(256), 0, st, C, R, a, activation);
        return check_launch("linear_forward_per_token");
    };
    // Wide K: quantise into a workspace, then the tiled GEMM (below).
    RowsArgs g = a;
    g.Aq = nullptr;  // the codes go to the workspace, which is 256-byte aligned
    const bool wide = use_gemm(g);
    const bool refused = fixed && noalloc_refuses(a, wide, fixed->cap);
    if (!refused && use_skinny(a)) {
        launch_skinny_i8(a, act_x2, st);
        return finish();
    }
    if (use_rows(a, IN_F32_TOKEN, false)) {
        launch_rows<false, IN_F32_TOKEN, OUT_EPI>(a, act_x2, st);
        return finish();
    }
    // The split form takes a workspace: not where the no-allocation entry
    // point's callers rely on the shape using none, nor for a capture that the
    // one-pass kernel can serve.
    const bool one_pass = use_token_gemm(a);
    // On the per-thread default stream a workspace costs an allocation and a
    // free per call: shapes that need none keep to that.
    const bool none_taken = (fixed || st == hipStreamPerThread) && noalloc_scratch_free(a, wide);
    const bool split = wide && split_faster(a) && !none_taken && (fixed || !stream_capturing(st));
    if (!refused && one_pass && !split) {
        launch_token_i8(a, act_x2, st);
        return finish();
    }
    // Split path: quantise into a workspace, then the product.
    // Workspace: codes, then M scales; for the tiled GEMM, M row code sums
    // from the same quantise pass when zero points may be nonzero, and N
    // weight-row byte sums when the formula takes a caller's sum_W.
    const size_t codes = static_cast<size_t>(M) * a.K;
    const bool want_sums = wide && a.zpW;
    const bool want_colsum = wide && a.formula == F_ROW_VNNI && a.sumW;
    const size_t n_sums = split_sums(a, wide);
    const size_t codes16 = ((codes + 15) / 16) * 16;
    if (fixed) {
        // Codes, then (with no scale_A_out) M scales, then the sums; every
        // region is written by the quantise launch before the product reads it.
        const size_t need = noalloc_need(a, wide);
        if (need > fixed->cap)
            return set_error(NFLOW_INVALID_ARG, std::string(fixed->what) + ": this shape needs " +
                                                    std::to_string(need) + " bytes of scratch, more than the " +
                                                    std::to_string(fixed->cap) + " the library holds (split the rows)");
        void* base = nullptr;
        std::unique_lock<std::mutex> hold;   // until the product is launched (end of scope)
        if (int rc = noalloc_scratch_address(&base, &hold)) return rc;
        uint8_t* q = static_cast<uint8_t*>(base);
        float* sc = scale_A_out ? scale_A_out : reinterpret_cast<float*>(q + codes16);
        int32_t* sums0 = reinterpret_cast<int32_t*>(q + codes16 + (scale_A_out ? 0 : static_cast<size_t>(M) * sizeof(float)));
        int32_t* sums = want_sums ? sums0 : nullptr;
        int32_t* colsum = want_colsum ? sums0 + (want_sums ? M : 0) : nullptr;
        launch_quantise_token<false>(A, M, a.K, q, sc, sums, st, CodeSums{a.W, a.N, a.K, colsum});
        a.Aq = q;
        a.scale_in = sc;
        a.sum_in = sums;
        a.colsum_in = colsum;
        if (wide) launch_gemm<OUT_EPI>(a, act_x2, st);
        else if (rows_ok(a, IN_CODES)) launch_rows<false, IN_CODES, OUT_EPI>(a, act_x2, st);
        else launch_generic<false, OUT_EPI>(a, act_x2, st);
        return finish();
    }
    Scratch ws(codes + 16 + static_cast<size_t>(M) * sizeof(float) + n_sums * sizeof(int32_t), st);
    if (ws.err != hipSuccess && one_pass) {
        (void)hipGetLastError();
        launch_token_i8(a, act_x2, st);
        return finish();
    }
    if (ws.err != hipSuccess) return set_error(NFLOW_INTERNAL, "linear_forward_per_token: workspace allocation failed");
    uint8_t* q = static_cast<uint8_t*>(ws.p);
    float* sc = reinterpret_cast<float*>(q + codes16);
    int32_t* sums = want_sums ? reinterpret_cast<int32_t*>(sc + M) : nullptr;
    int32_t* colsum = want_colsum ? reinterpret_cast<int32_t*>(sc + M) + (want_sums ? M : 0) : nullptr;
    launch_quantise_token<false>(A, M, a.K, q, sc, sums, st, CodeSums{a.W, a.N, a.K, colsum});
    if (scale_A_out) (void)hipMemcpyAsync(scale_A_out, sc, sizeof(float) * M, hipMemcpyDeviceToDevice, st);
    a.Aq = q;
    a.scale_in = sc;
    a.sum_in = sums;
    a.colsum_in = colsum;
    if (wide) launch_gemm<OUT_EPI>(a, act_x2, st);
    else if (rows_ok(a, IN_CODES)) launch_rows<false, IN_CODES, OUT_EPI>(a, act_x2, st);
    else launch_generic<false, OUT_EPI>(a, act_x2, st);
    return finish();
}

}  // namespace nfq

extern "C" {

int nflow_int8_linear_forward_per_token(const nflow_int8_linear_params* p, int64_t M,
                                        const float* A, float* C, float* scale_A_out,
                                        int activation, void* stream) {
    clear_error();
    return int8_per_token(p, M, A, nullptr, C, scale_A_out, activation, nullptr, stream);
}

int nflow_int8_linear_forward_per_token_noalloc(const nflow_int8_linear_params* p, int64_t M,
                                                const float* A, float* C, float* scale_A_out,
                                                int activation, void* stream) {
    clear_error();
    FixedWs fixed{kNoAllocScratchBytes, "linear_forward_per_token_noalloc"};
    return int8_per_token(p, M, A, nullptr, C, scale_A_out, activation, nullptr, stream, &fixed);
}

int nflow_int8_fno_layer_per_token(const nflow_int8_linear_params* p, int64_t M, const float* h,
                                   const float* x1, float* y, float* scale_A_out, int activation,
                                   void* stream) {
    clear_error();
    return int8_per_token(p, M, h, x1, y, scale_A_out, activation, nullptr, stream);
}

int nflow_int8_fno_layer_per_token_x2q(const nflow_int8_linear_params* p, int64_t M, const float* h,
                                       const float* x1, float* y, float* scale_A_out, int activation,
                                       const nflow_x2_quant* x2q, void* stream) {
    clear_error();
    return int8_per_token(p, M, h, x1, y, scale_A_out, activation, x2q, stream);
}

int nflow_int8_gemm_i32(const int8_t* A_q, const int8_t* W_q, int64_t M, int N, int K, int32_t* C,
                        void* stream) {
    clear_error();
    if (!A_q || !W_q || !C) return set_error(NFLOW_INVALID_ARG, "gemm_i32: null pointer");
    if (N <= 0 || K <= 0) return set_error(NFLOW_INVALID_ARG, "gemm_i32: bad dims");
    if (M <= 0) return NFLOW_OK;
    RowsArgs a{};
    a.Aq = reinterpret_cast<const uint8_t*>(A_q);
    a.M = M;
    a.K = K;
    a.N = N;
    a.W = reinterpret_cast<const uint8_t*>(W_q);
    a.kb_dot = (K + 63) / 64;
    a.C = C;
    if (use_gemm(a)) launch_gemm<OUT_RAW>(a, ACT_NONE, as_stream(stream));
    else if (rows_ok(a, IN_CODES)) launch_rows<false, IN_CODES, OUT_RAW>(a, ACT_NONE, as_stream(stream));
    else launch_generic<false, OUT_RAW>(a, ACT_NONE, as_stream(stream));
    return check_launch("gemm_i32");
}

int nflow_int8_linear_forward_quantised(const nflow_int8_linear_params* p, int64_t M,
                                        const int8_t* A_q, const float* scale_A, float* C,
                                        int activation, void* stream) {
    clear_error();
    if (!A_q || !scale_A || !C || !p || !p->W_int8 || !p->scale_W)
        return set_error(NFLOW_INVALID_ARG, "linear_forward_quantised: null input/output");
    if (p->in_features <= 0 || p->out_features <= 0)
        return set_error(NFLOW_INVALID_ARG, "linear_forward_quantised: bad feature dims");
    if (!valid_act(activation))
        return set_error(NFLOW_INVALID_ARG, "linear_forward_quantised: unknown activation");
    if (M <= 0) return NFLOW_OK;
    RowsArgs a{};
    a.Aq = reinterpret_cast<const uint8_t*>(A_q);
    a.scale_in = scale_A;
    a.M = M;
    a.K = p->in_features;
    a.N = p->out_features;
    a.W = reinterpret_cast<const uint8_t*>(p->W_int8);
    a.sW = p->scale_W;
    a.zpW = p->zp_W;
    a.bias = p->bias;
    a.sumW = p->sum_W_per_row;
    a.zp_A = 0;
    a.formula = formula_row(a.K);
    a.kb_dot = kb_dot_for(a.formula, a.K);
    a.C = C;
    hipStream_t st = as_stream(stream);
    if (use_gemm(a)) {
        // Without zero points a caller's sum_W only needs the weight-row
        // byte sums (a pre-pass) to keep the GEMM on its LDS-DMA kernel.
        if (!a.zpW && a.formula == F_ROW_VNNI && a.sumW) {
            Scratch ws(static_cast<size_t>(a.N) * sizeof(int32_t), st);
            if (ws.err != hipSuccess)
                return set_error(NFLOW_INTERNAL, "linear_forward_quantised: workspace allocation failed");
            int32_t* colsum = static_cast<int32_t*>(ws.p);
            hipLaunchKernelGGL(k_code_sums, dim3(grid_for(a.N, 16, 4)), dim3(256), 0, st, CodeSums{a.W, a.N, a.K, colsum});
            a.colsum_in = colsum;
            launch_gemm<OUT_EPI>(a, activation, st);
            return check_launch("linear_forward_quantised");
        }
        launch_gemm<OUT_EPI>(a, activation, st);
    } else if (rows_ok(a, IN_CODES)) {
        launch_rows<false, IN_CODES, OUT_EPI>(a, activation, st);
    } else {
        launch_generic<false, OUT_EPI>(a, activation, st);
    }
    return check_launch("linear_forward_quantised");
}

int nflow_fp8_e4m3_to_bits(const float* in, uint8_t* out, int64_t n, void* stream) {
    clear_error();
    if (!in || !out) return set_error(NFLOW_INVALID_ARG, "fp8_e4m3_to_bits: null pointer");
    if (n <= 0) return NFLOW_OK;
    const int per = elem_per(n, aligned(in, 16) && aligned(out, 4));
    hipLaunchKernelGGL(k_e4m3_encode, elem_grid(n, per), dim3(256), 0, as_stream(stream), in, out, n, per);
    return check_launch("fp8_e4m3_to_bits");
}

int nflow_fp8_e4m3_from_bits(const uint8_t* in, float* out, int64_t n, void* stream) {
    clear_error();
    if (!in || !out) return set_error(NFLOW_INVALID_ARG, "fp8_e4m3_from_bits: null pointer");
    if (n <= 0) return NFLOW_OK;
    const int per = elem_per(n, aligned(in, 4) && aligned(out, 16));
    hipLaunchKernelGGL(k_e4m3_decode, elem_grid(n, per), dim3(256), 0, as_stream(stream), in, out, n, per);
    return check_launch("fp8_e4m3_from_bits");
}

int nflow_fp8_e4m3_fake_quant(const float* in, float scale, float* out, int64_t n, void* stream) {
    clear_error();
    if (!in || !out) return set_error(NFLOW_INVALID_ARG, "fp8_e4m3_fake_quant: null pointer");
    if (n <= 0) return NFLOW_OK;
    const int per = elem_per(n, aligned(in, 16) && aligned(out, 16));
    hipLaunchKernelGGL(k_fp8_fake_quant, elem_grid(n, per), dim3(256), 0, as_stream(stream), in, scale, out, n, per);
    return check_launch("fp8_e4m3_fake_quant");
}

int nflow_fp8_quantise_per_token(const float* A, int64_t M, int K, uint8_t* A_q, float* scale_A,
                                 void* stream) {
    clear_error();
    if (!A || !A_q || !scale_A) return set_error(NFLOW_INVALID_ARG, "fp8_quantise_per_token: null pointer");
    if (K <= 0) return set_error(NFLOW_INVALID_ARG, "fp8_quantise_per_token: K <= 0");
    if (M <= 0) return NFLOW_OK;
    launch_quantise_token<true>(A, M, K, A_q, scale_A, static_cast<int32_t*>(nullptr), as_stream(stream));
    return check_launch("fp8_quantise_per_token");
}

static int fp8_check(const nflow_fp8_linear_params* p, int act, const char* what) {
    if (!p || !p->W_e4m3 || !p->scale_W) return set_error(NFLOW_INVALID_ARG, std::string(what) + ": null input/output");
    if (p->in_features <= 0 || p->out_features <= 0)
        return set_error(NFLOW_INVALID_ARG, std::string(what) + ": bad feature dims");
    if (!valid_act(act)) return set_error(NFLOW_INVALID_ARG, std::string(what) + ": unknown activation");
    return NFLOW_OK;
}

}  // extern "C"

namespace nfq {

static int fp8_per_token(const nflow_fp8_linear_params* p, int64_t M, const float* A, const float* R,
                         float* C, float* scale_A_out, int activation, const nflow_x2_quant* xq,
                         void* stream) {
    if (!A || !C) return set_error(NFLOW_INVALID_ARG, "fp8_linear_forward_per_token: null input/output");
    int rc = fp8_check(p, activation, "fp8_linear_forward_per_token");
    if (rc) return rc;
    if (R && R == C) return set_error(NFLOW_INVALID_ARG, "fp8_fno_layer: x1 and y must be distinct buffers");
    RowsArgs a{};
    a.N = p->out_features;
    if (int rc2 = apply_x2q(a, xq, "fp8_fno_layer")) return rc2;
    if (M <= 0) return NFLOW_OK;
    hipStream_t st = as_stream(stream);
    a.A = A;
    a.M = M;
    a.K = p->in_features;
    a.W = p->W_e4m3;
    a.sW = p->scale_W;
    a.bias = p->bias;
    a.kb_dot = (a.K + 63) / 64;
    a.C = C;
    a.scale_out = scale_A_out;
    if (rows64_ok(a) && (!R || aligned(R, 16)) && !path_flag(kernel_path().no_rows64)) {
        a.residual = R;
        launch_rows64<true>(a, activation, st);
        return check_launch("fp8_linear_forward_per_token");
    }
    const bool post = R || a.xq_kind;
    const int act_x2 = post ? static_cast<int>(ACT_NONE) : activation;
    auto finish = [&]() {
        if (post) hipLaunchKernelGGL(k_fno_post, dim3(grid_for(M, 1, 16)), dim3(256), 0, st, C, R, a, activation);
        return check_launch("fp8_linear_forward_per_token");
    };
    if (use_skinny(a)) {
        launch_skinny_fp8(a, act_x2, st);
        return finish();
    }
    if (use_rows(a, IN_F32_TOKEN, true)) {
        launch_rows<true, IN_F32_TOKEN, OUT_EPI>(a, act_x2, st);
        return finish();
    }
    // K a multiple of 64, at least 512: quantise, then the tiled GEMM, where
    // that is the faster form.
    RowsArgs g = a;
    g.Aq = nullptr;  // the codes go to the workspace, which is 256-byte aligned
    const bool wide = a.K >= 512 && use_gemm(g);
    if (use_token_gemm(a) && !(wide && fp8_split_faster(a) && !stream_capturing(st))) {
        launch_token_fp8(a, act_x2, st);
        return finish();
    }
    const size_t codes = static_cast<size_t>(M) * a.K;
    Scratch ws(codes + 16 + static_cast<size_t>(M) * sizeof(float), st);
    if (ws.err != hipSuccess && use_token_gemm(a)) {
        (void)hipGetLastError();
        launch_token_fp8(a, act_x2, st);
        return finish();
    }
    if (ws.err != hipSuccess) return set_error(NFLOW_INTERNAL, "fp8_linear_forward_per_token: workspace allocation failed");
    uint8_t* q = static_cast<uint8_t*>(ws.p);
    float* sc = reinterpret_cast<float*>(q + ((codes + 15) / 16) * 16);
    launch_quantise_token<true>(A, M, a.K, q, sc, static_cast<int32_t*>(nullptr), st);
    if (scale_A_out) (void)hipMemcpyAsync(scale_A_out, sc, sizeof(float) * M, hipMemcpyDeviceToDevice, st);
    a.Aq = q;
    a.scale_in = sc;
    if (wide) launch_gemm_fp8<OUT_EPI>(a, act_x2, st);
    else if (rows_ok(a, IN_CODES)) launch_rows<true, IN_CODES, OUT_EPI>(a, act_x2, st);
    else launch_generic<true, OUT_EPI>(a, act_x2, st);
    return finish();
}

}  // namespace nfq

extern "C" {

int nflow_fp8_linear_forward_per_token(const nflow_fp8_linear_params* p, int64_t M, const float* A,
                                       float* C, float* scale_A_out, int activation, void* stream) {
    clear_error();
    return fp8_per_token(p, M, A, nullptr, C, scale_A_out, activation, nullptr, stream);
}

int nflow_fp8_fno_layer_per_token(const nflow_fp8_linear_params* p, int64_t M, const float* h,
                                  const float* x1, float* y, float* scale_A_out, int activation,
                                  void* stream) {
    clear_error();
    return fp8_per_token(p, M, h, x1, y, scale_A_out, activation, nullptr, stream);
}

int nflow_fp8_fno_layer_per_token_x2q(const nflow_fp8_linear_params* p, int64_t M, const float* h,
                                      const float* x1, float* y, float* scale_A_out, int activation,
                                      const nflow_x2_quant* x2q, void* stream) {
    clear_error();
    return fp8_per_token(p, M, h, x1, y, scale_A_out, activation, x2q, stream);
}

int nflow_fp8_gemm_f32(const uint8_t* A_q, const uint8_t* W_q, int64_t M, int N, int K, float* C,
                       void* stream) {
    clear_error();
    if (!A_q || !W_q || !C) return set_error(NFLOW_INVALID_ARG, "fp8_gemm_f32: null pointer");
    if (N <= 0 || K <= 0) return set_error(NFLOW_INVALID_ARG, "fp8_gemm_f32: bad dims");
    if (M <= 0) return NFLOW_OK;
    RowsArgs a{};
    a.Aq = A_q;
    a.M = M;
    a.K = K;
    a.N = N;
    a.W = W_q;
    a.kb_dot = (K + 63) / 64;
    a.C = C;
    if (use_gemm(a)) launch_gemm_fp8<OUT_RAW>(a, ACT_NONE, as_stream(stream));
    else if (rows_ok(a, IN_CODES)) launch_rows<true, IN_CODES, OUT_RAW>(a, ACT_NONE, as_stream(stream));
    else launch_generic<true, OUT_RAW>(a, ACT_NONE, as_stream(stream));
    return check_launch("fp8_gemm_f32");
}

int nflow_fp8_linear_forward_quantised(const nflow_fp8_linear_params* p, int64_t M,
                                       const uint8_t* A_q, const float* scale_A, float* C,
                                       int activation, void* stream) {
    clear_error();
    if (!A_q || !scale_A || !C) return set_error(NFLOW_INVALID_ARG, "fp8_linear_forward_quantised: null input/output");
    int rc = fp8_check(p, activation, "fp8_linear_forward_quantised");
    if (rc) return rc;
    if (M <= 0) return NFLOW_OK;
    RowsArgs a{};
    a.Aq = A_q;
    a.scale_in = scale_A;
    a.M = M;
    a.K = p->in_features;
    a.N = p->out_features;
    a.W = p->W_e4m3;
    a.sW = p->scale_W;
    a.bias = p->bias;
    a.kb_dot = (a.K + 63) / 64;
    a.C = C;
    if (use_gemm(a)) launch_gemm_fp8<OUT_EPI>(a, activation, as_stream(stream));
    else if (rows_ok(a, IN_CODES)) launch_rows<true, IN_CODES, OUT_EPI>(a, activation, as_stream(stream));
    else launch_generic<true, OUT_EPI>(a, activation, as_stream(stream));
    return check_launch("fp8_linear_forward_quantised");
}

}  // extern "C"

namespace nfq {

// ---------------------------------------------------------------------------
// 8-bit-output layers and the per-token layer chain
// ---------------------------------------------------------------------------

// Row-maxima exchange state of the 8-bit-output kernel, per (device,
// stream): the published words (zeroed when allocated; every launch tags its
// words with a new epoch, so a word of an earlier launch never reads as
// fresh) and a fault word, set by a launch whose wait for the other blocks
// of a row tile timed out.  Calls on one stream run in order; calls on
// different streams use different words.  The words grow with the largest M
// (freed and reallocated in stream order) and live until the process ends.
struct ChainState {
    std::mutex mu;
    uint64_t* part = nullptr;
    int64_t rows_cap = 0;
    uint32_t* fault = nullptr;
};

static ChainState* chain_state(int dev, hipStream_t st) {
    static std::mutex map_mu;
    static std::map<std::pair<int, uintptr_t>, std::unique_ptr<ChainState>>* map =
        new std::map<std::pair<int, uintptr_t>, std::unique_ptr<ChainState>>();
    std::lock_guard<std::mutex> g(map_mu);
    auto& e = (*map)[{dev, reinterpret_cast<uintptr_t>(st)}];
    if (!e) e.reset(new ChainState);
    return e.get();
}

// A nonzero tag no earlier launch of this process used (wraps after 2^32 - 1
// launches).
static uint32_t next_chain_epoch() {
    static std::atomic<uint32_t> e{0};
    uint32_t v;
    do v = e.fetch_add(1, std::memory_order_relaxed) + 1; while (v == 0);
    return v;
}

// A wave waits at most this long (ticks of the 100 MHz clock: 2 s) for the
// other blocks of its row tile; they run concurrently, so a timeout means
// they could not be scheduled.
constexpr int64_t kChainSpinTicks = 200000000;
constexpr int kChainSlots = 8;   // published words per row, at most (128-column tiles, N <= 1024)

// Words for M rows (and the fault word) in cs, allocated on stream st.
static int chain_words(ChainState* cs, int64_t M, hipStream_t st) {
    const int64_t rows = ((M + 127) / 128) * 128;
    if (!cs->fault) {
        if (hipMallocAsync(reinterpret_cast<void**>(&cs->fault), 256, st) != hipSuccess) {
            cs->fault = nullptr;
            return set_error(NFLOW_INTERNAL, "chain: fault word allocation failed");
        }
        if (hipMemsetAsync(cs->fault, 0, 256, st) != hipSuccess) return set_error(NFLOW_INTERNAL, "chain: memset failed");
    }
    if (rows > cs->rows_cap) {
        if (cs->part) (void)hipFreeAsync(cs->part, st);
        cs->part = nullptr;
        cs->rows_cap = 0;
        const int64_t want = std::max<int64_t>(rows, 4096);
        const size_t bytes = static_cast<size_t>(want) * kChainSlots * sizeof(uint64_t);
        if (hipMallocAsync(reinterpret_cast<void**>(&cs->part), bytes, st) != hipSuccess) {
            cs->part = nullptr;
            return set_error(NFLOW_INTERNAL, "chain: row-maxima allocation failed");
        }
        if (hipMemsetAsync(cs->part, 0, bytes, st) != hipSuccess) return set_error(NFLOW_INTERNAL, "chain: memset failed");
        cs->rows_cap = want;
    }
    return NFLOW_OK;
}

// The chain entry points refuse a capturing stream before any allocation or
// launch: the fused kernel's row-maxima words would be allocated and cleared
// inside the graph and a replay would reuse its launch's epoch (an earlier
// replay's words reading as fresh); the layer-by-layer route allocates its
// buffers inside the graph, and a graph captured that way (both entry
// points, 20000 rows) took an illegal memory access on its first replay, for
// a reason not found in this library.
//
// Whether calls on stream st may use the fused 8-bit-output kernel: not on
// the per-thread default stream, whose one handle names a different stream
// in each host thread, so concurrent launches would share the row-maxima
// words.  Those calls take the layer-by-layer path (the same bits).
static bool chain_stream_ok(hipStream_t st) { return st != hipStreamPerThread; }

// Whether a layer takes the fused 8-bit-output kernel: symmetric weights
// (no zero points, no caller sum_W: the integer terms of the formula are 0),
// K = 1024, N a multiple of 256 up to 1024, 16-byte aligned codes.
static bool chain_layer_ok(const nflow_int8_linear_params* p) {
    return !p->zp_W && !p->sum_W_per_row && p->in_features == 1024 && p->out_features >= 256 &&
           p->out_features <= 1024 && p->out_features % 256 == 0 && aligned(p->W_int8, 16);
}

// One fused layer on stream st with cs's words (cs locked by the caller).
static void chain_launch(const nflow_int8_linear_params* p, int64_t M, const uint8_t* Aq, const float* sA,
                         uint8_t* Cq, float* sC, int act, hipStream_t st, ChainState* cs) {
    ChainArgs c{};
    c.Aq = Aq;
    c.scale_in = sA;
    c.M = M;
    c.K = p->in_features;
    c.N = p->out_features;
    c.W = reinterpret_cast<const uint8_t*>(p->W_int8);
    c.sW = p->scale_W;
    c.bias = p->bias;
    c.Cq = Cq;
    c.scale_out = sC;
    c.part = cs->part;
    c.fault = cs->fault;
    c.epoch = next_chain_epoch();
    c.spin_limit = kChainSpinTicks;
    launch_chain(c, act, st);
}

// Codes + row scales -> fp32 (M, N) through the LinearForward formula with
// zp_A = 0 (the product of nflow_int8_linear_forward_quantised for
// symmetric layers and for those the tiled kernel forms the byte sums of).
static void codes_to_f32(const nflow_int8_linear_params* p, int64_t M, const uint8_t* Aq, const float* sA,
                         float* C, int act, hipStream_t st) {
    RowsArgs a{};
    a.Aq = Aq;
    a.scale_in = sA;
    a.M = M;
    a.K = p->in_features;
    a.N = p->out_features;
    a.W = reinterpret_cast<const uint8_t*>(p->W_int8);
    a.sW = p->scale_W;
    a.zpW = p->zp_W;
    a.bias = p->bias;
    a.sumW = p->sum_W_per_row;
    a.zp_A = 0;
    a.formula = formula_row(a.K);
    a.kb_dot = kb_dot_for(a.formula, a.K);
    a.C = C;
    if (use_gemm(a)) launch_gemm<OUT_EPI>(a, act, st);
    else if (rows_ok(a, IN_CODES)) launch_rows<false, IN_CODES, OUT_EPI>(a, act, st);
    else launch_generic<false, OUT_EPI>(a, act, st);
}

static int check_layer(const nflow_int8_linear_params* p, int act, const char* what) {
    if (!p || !p->W_int8 || !p->scale_W) return set_error(NFLOW_INVALID_ARG, std::string(what) + ": null layer parameters");
    if (p->in_features <= 0 || p->out_features <= 0)
        return set_error(NFLOW_INVALID_ARG, std::string(what) + ": bad feature dims");
    if (!valid_act(act)) return set_error(NFLOW_INVALID_ARG, std::string(what) + ": unknown activation");
    return NFLOW_OK;
}

}  // namespace nfq

extern "C" {

int nflow_int8_linear_forward_codes(const nflow_int8_linear_params* p, int64_t M, const int8_t* A_q,
                                    const float* scale_A, int8_t* C_q, float* scale_C, int activation,
                                    void* stream) {
    clear_error();
    if (int rc = check_layer(p, activation, "linear_forward_codes")) return rc;
    if (!A_q || !scale_A || !C_q || !scale_C) return set_error(NFLOW_INVALID_ARG, "linear_forward_codes: null input/output");
    if (M <= 0) return NFLOW_OK;
    hipStream_t st = as_stream(stream);
    if (stream_capturing(st))
        return set_error(NFLOW_UNSUPPORTED_OP, "linear_forward_codes: not available under graph capture (use "
                                               "nflow_int8_linear_forward_per_token_noalloc)");
    const uint8_t* aq = reinterpret_cast<const uint8_t*>(A_q);
    uint8_t* cq = reinterpret_cast<uint8_t*>(C_q);
    if (chain_layer_ok(p) && aligned(aq, 16) && aligned(cq, 4) && chain_stream_ok(st)) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return set_error(NFLOW_INTERNAL, "linear_forward_codes: hipGetDevice failed");
        ChainState* cs = chain_state(dev, st);
        std::lock_guard<std::mutex> lock(cs->mu);
        if (int rc = chain_words(cs, M, st)) return rc;
        chain_launch(p, M, aq, scale_A, cq, scale_C, activation, st, cs);
        return check_launch("linear_forward_codes");
    }
    // Other layers: the fp32 output into a stream-ordered buffer, then the
    // per-token quantise (the same bits).
    float* tmp = nullptr;
    const size_t bytes = static_cast<size_t>(M) * p->out_features * sizeof(float);
    if (hipMallocAsync(reinterpret_cast<void**>(&tmp), bytes, st) != hipSuccess)
        return set_error(NFLOW_INTERNAL, "linear_forward_codes: workspace allocation failed");
    int rc = nflow_int8_linear_forward_quantised(p, M, A_q, scale_A, tmp, activation, stream);
    if (rc == NFLOW_OK) {
        launch_quantise_token<false>(tmp, M, p->out_features, cq, scale_C, nullptr, st);
        rc = check_launch("linear_forward_codes");
    }
    (void)hipFreeAsync(tmp, st);
    return rc;
}

int nflow_int8_mlp_forward_per_token(const nflow_int8_linear_params* layers, const int* activations,
                                     int n_layers, int64_t M, const float* x, float* y, void* stream) {
    clear_error();
    if (!layers || !activations || n_layers <= 0) return set_error(NFLOW_INVALID_ARG, "mlp_forward_per_token: no layers");
    if (!x || !y) return set_error(NFLOW_INVALID_ARG, "mlp_forward_per_token: null input/output");
    for (int l = 0; l < n_layers; ++l) {
        if (int rc = check_layer(&layers[l], activations[l], "mlp_forward_per_token")) return rc;
        if (l > 0 && layers[l].in_features != layers[l - 1].out_features)
            return set_error(NFLOW_SHAPE_MISMATCH, "mlp_forward_per_token: layer " + std::to_string(l) +
                                                       " in_features != the previous layer's out_features");
    }
    if (M <= 0) return NFLOW_OK;
    hipStream_t st = as_stream(stream);
    if (stream_capturing(st))
        return set_error(NFLOW_UNSUPPORTED_OP, "mlp_forward_per_token: not available under graph capture (use "
                                               "nflow_int8_linear_forward_per_token_noalloc per layer)");
    if (n_layers == 1) return int8_per_token(&layers[0], M, x, nullptr, y, nullptr, activations[0], nullptr, stream);
    // Fused: every layer symmetric, every layer but the last on the
    // 8-bit-output kernel (K = 1024, so every hidden width is 1024), and
    // rows enough for two 128 x 256 tiles per CU: with one tile per CU the
    // 8-bit-output kernel's last row-maxima exchange is not overlapped
    // (measured at 4096 rows, K = N = 1024: 17.9 us against 11.2 us for the
    // fp32-output product, more than the quantise launch it saves).
    bool fused = aligned(x, 16) && !layers[n_layers - 1].zp_W && !layers[n_layers - 1].sum_W_per_row &&
                 ((M + 127) / 128) * 4 >= 2 * static_cast<int64_t>(num_cus()) && chain_stream_ok(st);
    for (int l = 0; l < n_layers - 1; ++l) fused = fused && chain_layer_ok(&layers[l]);
    if (fused) {
        const size_t codes = static_cast<size_t>(M) * 1024;
        const size_t codes16 = ((codes + 255) / 256) * 256;
        const size_t sc = ((static_cast<size_t>(M) * sizeof(float) + 255) / 256) * 256;
        Scratch ws(2 * codes16 + 2 * sc, st);
        if (ws.err != hipSuccess) return set_error(NFLOW_INTERNAL, "mlp_forward_per_token: workspace allocation failed");
        uint8_t* q[2] = {static_cast<uint8_t*>(ws.p), static_cast<uint8_t*>(ws.p) + codes16};
        float* s[2] = {reinterpret_cast<float*>(q[1] + codes16), reinterpret_cast<float*>(q[1] + codes16 + sc)};
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return set_error(NFLOW_INTERNAL, "mlp_forward_per_token: hipGetDevice failed");
        ChainState* cs = chain_state(dev, st);
        std::lock_guard<std::mutex> lock(cs->mu);
        if (int rc = chain_words(cs, M, st)) return rc;
        launch_quantise_token<false>(x, M, 1024, q[0], s[0], nullptr, st);
        int cur = 0;
        for (int l = 0; l < n_layers - 1; ++l) {
            chain_launch(&layers[l], M, q[cur], s[cur], q[cur ^ 1], s[cur ^ 1], activations[l], st, cs);
            cur ^= 1;
        }
        codes_to_f32(&layers[n_layers - 1], M, q[cur], s[cur], y, activations[n_layers - 1], st);
        return check_launch("mlp_forward_per_token");
    }
    // Layer by layer through fp32 activations in two buffers of the stream's
    // second workspace slot (each layer's own workspace is slot 0).
    int width = 0;
    for (int l = 0; l < n_layers - 1; ++l) width = std::max(width, layers[l].out_features);
    const size_t hb = ((static_cast<size_t>(M) * width * sizeof(float) + 255) / 256) * 256;
    Scratch hs(2 * hb, st, 1);
    if (hs.err != hipSuccess) return set_error(NFLOW_INTERNAL, "mlp_forward_per_token: workspace allocation failed");
    float* h[2] = {static_cast<float*>(hs.p), reinterpret_cast<float*>(static_cast<uint8_t*>(hs.p) + hb)};
    int rc = NFLOW_OK;
    const float* in = x;
    for (int l = 0; l < n_layers && rc == NFLOW_OK; ++l) {
        float* out = l == n_layers - 1 ? y : h[l & 1];
        rc = int8_per_token(&layers[l], M, in, nullptr, out, nullptr, activations[l], nullptr, stream);
        in = out;
    }
    return rc;
}

int nflow_release_stream_workspace(void* stream) {
    clear_error();
    hipStream_t st = as_stream(stream);
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return set_error(NFLOW_INTERNAL, "release_stream_workspace: hipGetDevice failed");
    for (int slot = 0; slot < 2; ++slot) {
        WsEntry* e = ws_entry(dev, st, slot);
        std::lock_guard<std::mutex> lock(e->mu);
        if (e->p) (void)hipFreeAsync(e->p, st);
        e->p = nullptr;
        e->cap = 0;
    }
    ChainState* cs = chain_state(dev, st);
    std::lock_guard<std::mutex> lock(cs->mu);
    if (cs->part) (void)hipFreeAsync(cs->part, st);
    if (cs->fault) (void)hipFreeAsync(cs->fault, st);
    cs->part = nullptr;
    cs->fault = nullptr;
    cs->rows_cap = 0;
    return check_launch("release_stream_workspace");
}

int nflow_debug_chain_faults(void* stream, uint32_t* faults) {
    clear_error();
    if (!faults) return set_error(NFLOW_INVALID_ARG, "debug_chain_faults: null output");
    *faults = 0;
    hipStream_t st = as_stream(stream);
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return set_error(NFLOW_INTERNAL, "debug_chain_faults: hipGetDevice failed");
    ChainState* cs = chain_state(dev, st);
    std::lock_guard<std::mutex> lock(cs->mu);
    if (!cs->fault) return NFLOW_OK;
    uint32_t v = 0;
    if (hipMemcpyAsync(&v, cs->fault, sizeof(v), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess || hipMemsetAsync(cs->fault, 0, sizeof(uint32_t), st) != hipSuccess)
        return set_error(NFLOW_INTERNAL, "debug_chain_faults: copy failed");
    *faults = v;
    return NFLOW_OK;
}

}  // extern "C"
