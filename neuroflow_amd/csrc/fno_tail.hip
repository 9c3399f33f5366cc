// fno_tail.hip -- the FNO runtime's local linear (fp32 or INT8) with the layer
// tail, and the projection head, each in one launch, for widths other than 64
// (fno_rt.hip holds the width-64 forms).
//
// What bounds them: the ordered fp32 sums (one multiply and one add per term,
// W terms per output, no FMA: the reference's rounding) and the exact GELU
// on the VALU, and four activation streams of HBM.  Run as separate launches
// the local linear alone took 473 us at 262144 x 32 -> 32 (one thread per
// output, each reading its own weight row from the cache); here a thread
// holds its channel's weight row in W registers and reads the tile's h rows
// from LDS as broadcasts, and x2 never leaves the registers.  262144 points,
// width 32, log2 snap, GELU: linear + tail 473 + 58 -> 44.7 us (134 MB of
// streams: 27 us at the copy rate), projection head 473 + 25 + 13 -> 41.9 us;
// FNO2d 16 x 128 x 128 of width 32 2837 -> 396 us.
#include <hip/hip_runtime.h>

#include "fno_dev.h"

namespace nfq {

// Thread x of a block takes channel x % W of tokens x / W + (256 / W) q of a
// 32-token tile (256 - 256 % W threads compute).  W is a template parameter:
// the weight row's register indices and every offset are then constants.
template <int W>
struct TailShape {
    static constexpr int TT = 32;                    // tokens per tile
    static constexpr int RP = 256 / W;               // tokens per pass
    static constexpr int PER = (TT + RP - 1) / RP;   // passes
    static constexpr int HS = W + 4;                 // LDS row stride of the h tile (floats)
    static constexpr int NV = TT * W / 4;            // float4s of the h tile
    static constexpr int HV = (NV + 255) / 256;      // float4s per thread
    static constexpr int XV = (W + 7) / 8;           // channel-major elements per thread
};

// The reference Linear's sum (fno.cpp:69-79): the first W - W % 8 products
// rounded and added in order, the rest fused.
template <int W>
__device__ __forceinline__ float tail_dot(const float* hr, const float (&wr)[W], float acc) {
    constexpr int PLAIN = W - W % 8;
#pragma unroll
    for (int p = 0; p < W; p += 4) {
        const v4f h = *reinterpret_cast<const v4f*>(hr + p);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = lin_step(acc, h[e], wr[p + e], p < PLAIN);
    }
    return acc;
}

template <int W>
__device__ __forceinline__ void tail_weights(const float* w, float (&wr)[W]) {
#pragma unroll
    for (int p = 0; p < W; p += 4) {
        const v4f q = *reinterpret_cast<const v4f*>(w + p);
#pragma unroll
        for (int e = 0; e < 4; ++e) wr[p + e] = q[e];
    }
}

template <int W, int KIND, int ACT, int FQN>
__global__ __launch_bounds__(256) void k_linear_tail_w(PostArgs a, const float* Wl, const float* bl) {
    using S = TailShape<W>;
    __shared__ float tx1[W][S::TT + 1];
    __shared__ __attribute__((aligned(16))) float th[S::TT * S::HS];
    __shared__ float thr_x2[16], thr_next[16];
    const int n = a.n;                  // n % 32 == 0 (linear_tail_w_ok)
    if (threadIdx.x < 15) thr_x2[threadIdx.x] = a.thr[threadIdx.x];
    stage_steps(thr_next, a.fq_next.thr);
    const ScaleInv inv_x2 = scale_inv(a.scale), inv_next = scale_inv(a.fq_next.scale);
    const int tid = threadIdx.x;
    const int cm = tid / S::TT, tm = tid % S::TT;            // channel-major: channel, token
    const int tk = tid / W, ck = tid % W;                    // token-major: token, channel
    const bool live = tid < S::RP * W;
    float wr[W];
    tail_weights<W>(Wl + ck * W, wr);
    const float bj = bl ? bl[ck] : 0.0f;
    const int64_t o1 = static_cast<int64_t>(cm) * n + tm, d1 = static_cast<int64_t>(8) * n;
    Tile tl;
    for (int64_t id = blockIdx.x; tile_of<S::TT>(id, a.samples, n, W, tl); id += gridDim.x) {
        const int64_t cb = tl.s * W * static_cast<int64_t>(n) + tl.t0 + o1;
        const int64_t tb = (tl.s * n + tl.t0) * W;
        v4f hv[S::HV];
#pragma unroll
        for (int q = 0; q < S::HV; ++q)
            if (S::NV % 256 == 0 || tid + 256 * q < S::NV) hv[q] = *reinterpret_cast<const v4f*>(a.h + tb + 4 * (tid + 256 * q));
        float xv[S::XV];
#pragma unroll
        for (int q = 0; q < S::XV; ++q)
            if (W % 8 == 0 || cm + 8 * q < W) xv[q] = a.x1c[cb + q * d1];
#pragma unroll
        for (int q = 0; q < S::HV; ++q) {
            const int i = tid + 256 * q;
            if (S::NV % 256 == 0 || i < S::NV) *reinterpret_cast<v4f*>(th + (i / (W / 4)) * S::HS + 4 * (i % (W / 4))) = hv[q];
        }
#pragma unroll
        for (int q = 0; q < S::XV; ++q)
            if (W % 8 == 0 || cm + 8 * q < W) tx1[cm + 8 * q][tm] = xv[q];
        __syncthreads();
        float v[S::PER];
#pragma unroll
        for (int q = 0; q < S::PER; ++q) {
            const int t = tk + S::RP * q;
            if (S::TT % S::RP != 0 && t >= S::TT) continue;
            if (!live) continue;
            const float acc = tail_dot<W>(th + t * S::HS, wr, bj);
            v[q] = post_element<KIND, ACT, FQN>(tx1[ck][t], acc, a, inv_x2, inv_next, thr_x2, thr_next, 0.0f, 0.0f);
            tx1[ck][t] = v[q];
        }
#pragma unroll
        for (int q = 0; q < S::PER; ++q) {
            const int t = tk + S::RP * q;
            if (live && (S::TT % S::RP == 0 || t < S::TT)) a.h[tb + t * W + ck] = v[q];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < S::XV; ++q)
            if (W % 8 == 0 || cm + 8 * q < W) a.hc[cb + q * d1] = tx1[cm + 8 * q][tm];
        __syncthreads();
    }
}

// The INT8 local linear (LinearForwardBatched + bias with the layer's
// per-tensor scale, as fno.cpp:529-536 runs it) and the tail on the same
// tiles: the h tile becomes codes in LDS, four per dword, a thread holds its
// channel's W weight codes in W / 4 registers, and an output's product is W / 4
// v_dot4 (exact in int32; at these widths fewer instructions than the moves an
// MFMA's operand layouts would take).  As two launches (the fixed-scale layer
// and the tail) an FNO1d of 4 layers, 256 x 1024 of width 32, ran 484 us; 310
// with this kernel (60 x 1024: 232 -> 149).
template <int W, int KIND, int ACT, int FQN>
__global__ __launch_bounds__(256) void k_layer_tail_w(LayerTailArgs la, int int_epi) {
    using S = TailShape<W>;
    constexpr int KQ = W / 4, CS = KQ + 1;           // code dwords per token, row stride
    const PostArgs& a = la.p;
    __shared__ float tx1[W][S::TT + 1];
    __shared__ uint32_t codes[S::TT * CS];
    __shared__ float thr_x2[16], thr_next[16];
    const int n = a.n;                  // n % 32 == 0 (layer_tail_w_ok)
    if (threadIdx.x < 15) thr_x2[threadIdx.x] = a.thr[threadIdx.x];
    stage_steps(thr_next, a.fq_next.thr);
    const ScaleInv inv_x2 = scale_inv(a.scale), inv_next = scale_inv(a.fq_next.scale);
    const float fixed_inv = 1.0f / la.sA;
    const bool fixed_fast = la.sA >= 0x1p-120f && la.sA <= 0x1p120f;
    const int tid = threadIdx.x;
    const int cm = tid / S::TT, tm = tid % S::TT;            // channel-major: channel, token
    const int tk = tid / W, ck = tid % W;                    // token-major: token, channel
    const bool live = tid < S::RP * W;
    uint32_t wq[KQ];
    int32_t sfull = 0;
#pragma unroll
    for (int q = 0; q < KQ; ++q) {
        wq[q] = reinterpret_cast<const uint32_t*>(la.W + ck * W)[q];
        sfull = sum_bytes_i8(wq[q], sfull);
    }
    const IntEpi epi = int_epi_consts(F_BATCHED, W, la.zpA, la.zpW ? la.zpW[ck] : 0, la.sumW ? la.sumW[ck] : 0,
                                      la.sumW != nullptr, sfull, sfull);
    const float sw = la.sW[ck], bj = la.bias ? la.bias[ck] : 0.0f;
    const int64_t o1 = static_cast<int64_t>(cm) * n + tm, d1 = static_cast<int64_t>(8) * n;
    Tile tl;
    for (int64_t id = blockIdx.x; tile_of<S::TT>(id, a.samples, n, W, tl); id += gridDim.x) {
        const int64_t cb = tl.s * W * static_cast<int64_t>(n) + tl.t0 + o1;
        const int64_t tb = (tl.s * n + tl.t0) * W;
        v4f hv[S::HV];
#pragma unroll
        for (int q = 0; q < S::HV; ++q)
            if (S::NV % 256 == 0 || tid + 256 * q < S::NV) hv[q] = *reinterpret_cast<const v4f*>(a.h + tb + 4 * (tid + 256 * q));
        float xv[S::XV];
#pragma unroll
        for (int q = 0; q < S::XV; ++q)
            if (W % 8 == 0 || cm + 8 * q < W) xv[q] = a.x1c[cb + q * d1];
#pragma unroll
        for (int q = 0; q < S::XV; ++q)
            if (W % 8 == 0 || cm + 8 * q < W) tx1[cm + 8 * q][tm] = xv[q];
#pragma unroll
        for (int q = 0; q < S::HV; ++q) {
            const int i = tid + 256 * q;
            if (S::NV % 256 == 0 || i < S::NV)
                codes[(i / KQ) * CS + i % KQ] = quant_i8_fixed4(hv[q], la.sA, fixed_inv, la.zpA, fixed_fast);
        }
        __syncthreads();
        float v[S::PER];
#pragma unroll
        for (int q = 0; q < S::PER; ++q) {
            const int t = tk + S::RP * q;
            if (S::TT % S::RP != 0 && t >= S::TT) continue;
            if (!live) continue;
            const uint32_t* cr = codes + t * CS;
            int32_t D = 0, SA = 0;
#pragma unroll
            for (int k = 0; k < KQ; ++k) D = __builtin_amdgcn_sdot4(static_cast<int>(cr[k]), static_cast<int>(wq[k]), D, false);
            float tv;
            if (int_epi) {
#pragma unroll
                for (int k = 0; k < KQ; ++k) SA = sum_bytes_i8(cr[k], SA);
                tv = int_epi_value_fixed(epi, D, SA);
            } else {
                tv = static_cast<float>(D);
            }
            const float x2 = dequant_bias(sw, la.sA, tv, bj);
            v[q] = post_element<KIND, ACT, FQN>(tx1[ck][t], x2, a, inv_x2, inv_next, thr_x2, thr_next, 0.0f, 0.0f);
            tx1[ck][t] = v[q];
        }
#pragma unroll
        for (int q = 0; q < S::PER; ++q) {
            const int t = tk + S::RP * q;
            if (live && (S::TT % S::RP == 0 || t < S::TT)) a.h[tb + t * W + ck] = v[q];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < S::XV; ++q)
            if (W % 8 == 0 || cm + 8 * q < W) a.hc[cb + q * d1] = tx1[cm + 8 * q][tm];
        __syncthreads();
    }
}

// The projection head (fno.cpp:662-698, :966-993): proj_q W -> W, its
// fake-quant FQQ and the activation, then proj_out W -> 1 (32 threads, one
// token each, the W activations in order) and its fake-quant.
template <int W, int ACT, int FQQ>
__global__ __launch_bounds__(256) void k_proj_tail_w(ProjArgs a) {
    using S = TailShape<W>;
    constexpr int QS = W + 1;
    constexpr int PLAIN = W - W % 8;
    __shared__ __attribute__((aligned(16))) float th[S::TT * S::HS];
    __shared__ float tq[S::TT * QS];
    __shared__ float wo_s[W];
    __shared__ float steps_q[16], steps_o[16];
    const int tid = threadIdx.x;
    if (tid < W) wo_s[tid] = a.Wo[tid];
    stage_steps(steps_q, a.fq_q.thr);
    stage_steps(steps_o, a.fq_o.thr);
    const ScaleInv inv_q = scale_inv(a.fq_q.scale), inv_o = scale_inv(a.fq_o.scale);
    const int tk = tid / W, ck = tid % W;
    const bool live = tid < S::RP * W;
    float wr[W];
    tail_weights<W>(a.Wq + ck * W, wr);
    const float bj = a.bq ? a.bq[ck] : 0.0f;
    const float bo = a.bo ? a.bo[0] : 0.0f;
    const int n = a.n;
    Tile tl;
    for (int64_t id = blockIdx.x; tile_of<S::TT>(id, a.samples, n, W, tl); id += gridDim.x) {
        const float* hs = a.h + (tl.s * a.rows_in + tl.t0) * W;
        v4f hv[S::HV];
#pragma unroll
        for (int q = 0; q < S::HV; ++q)
            if (S::NV % 256 == 0 || tid + 256 * q < S::NV) hv[q] = *reinterpret_cast<const v4f*>(hs + 4 * (tid + 256 * q));
#pragma unroll
        for (int q = 0; q < S::HV; ++q) {
            const int i = tid + 256 * q;
            if (S::NV % 256 == 0 || i < S::NV) *reinterpret_cast<v4f*>(th + (i / (W / 4)) * S::HS + 4 * (i % (W / 4))) = hv[q];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < S::PER; ++q) {
            const int t = tk + S::RP * q;
            if (S::TT % S::RP != 0 && t >= S::TT) continue;
            if (!live) continue;
            float acc = tail_dot<W>(th + t * S::HS, wr, bj);
            if constexpr (FQQ == 1) acc = x2_fake_quant_inv(acc, a.fq_q.scale, inv_q.inv, inv_q.ok, a.fq_q.zpf);
            else if constexpr (FQQ == 3) acc = log2_snap(acc, a.fq_q.scale, steps_q);
            if constexpr (ACT == RT_ACT_RELU) acc = acc < 0.0f ? 0.0f : acc;   // fno.cpp:37-40
            else if constexpr (ACT == RT_ACT_GELU) acc = gelu_fast<kGeluRefine>(acc);
            tq[t * QS + ck] = acc;
        }
        __syncthreads();
        if (tid < S::TT) {
            const float* qr = tq + tid * QS;
            float acc = bo;
#pragma unroll
            for (int j = 0; j < W; ++j) acc = lin_step(acc, qr[j], wo_s[j], j < PLAIN);
            if (a.fq_o.on == 1) acc = x2_fake_quant_inv(acc, a.fq_o.scale, inv_o.inv, inv_o.ok, a.fq_o.zpf);
            else if (a.fq_o.on == 3) acc = log2_snap(acc, a.fq_o.scale, steps_o);
            a.y[tl.s * n + tl.t0 + tid] = acc;
        }
        // tq is next written after the next tile's first barrier, which the
        // reading threads reach only after their sums.
    }
}

// Widths with an instantiation: 16 to 48 in steps of 8, and 20.  The kernels
// hold for any multiple of 4 below 64; the others have not been instantiated or
// measured and keep the separate launches, as does the per-position x2
// fake-quant (KIND 2) at every width but 64.  The rest of the conditions are
// the width-64 forms': whole 32-token tiles, ReLU or GELU, the fake-quants.
static bool width_ok(int w) { return w == 16 || w == 20 || w == 24 || w == 32 || w == 40 || w == 48; }

bool linear_tail_w_ok(const PostArgs& p, const float* W) {
    return !path_flag(kernel_path().no_layer_tail) && width_ok(p.w) && p.n > 0 && p.n % 32 == 0 &&
           (p.act == RT_ACT_RELU || p.act == RT_ACT_GELU) && (p.fq_next.on == 0 || p.fq_next.on == 1) &&
           (p.kind == 0 || p.kind == 1 || p.kind == 3) && aligned(p.h, 16) && aligned(W, 16);
}

bool layer_tail_w_ok(const PostArgs& p, int in_features, int out_features) {
    return in_features == p.w && out_features == p.w && linear_tail_w_ok(p, nullptr);
}

bool proj_tail_w_ok(const ProjArgs& p) {
    const auto fq_ok = [](const FakeQuant& f) { return f.on == 0 || f.on == 1 || f.on == 3; };
    return !path_flag(kernel_path().no_layer_tail) && width_ok(p.w) && p.out_ch == 1 && p.n > 0 && p.n % 32 == 0 &&
           p.rows_in >= p.n &&
           fq_ok(p.fq_q) && fq_ok(p.fq_o) && (p.act == RT_ACT_RELU || p.act == RT_ACT_GELU) && aligned(p.h, 16) &&
           aligned(p.Wq, 16);
}

template <int W, int KIND, int ACT>
static void launch_lt_fqn(const PostArgs& a, const float* Wl, const float* b, unsigned grid, hipStream_t st) {
    if (a.fq_next.on == 1) hipLaunchKernelGGL((k_linear_tail_w<W, KIND, ACT, 1>), dim3(grid), dim3(256), 0, st, a, Wl, b);
    else hipLaunchKernelGGL((k_linear_tail_w<W, KIND, ACT, 0>), dim3(grid), dim3(256), 0, st, a, Wl, b);
}

template <int W, int KIND>
static void launch_lt_act(const PostArgs& a, const float* Wl, const float* b, unsigned grid, hipStream_t st) {
    if (a.act == RT_ACT_GELU) launch_lt_fqn<W, KIND, RT_ACT_GELU>(a, Wl, b, grid, st);
    else launch_lt_fqn<W, KIND, RT_ACT_RELU>(a, Wl, b, grid, st);
}

template <int W>
static void launch_lt(const PostArgs& a, const float* Wl, const float* b, hipStream_t st) {
    const unsigned grid = grid_for(tile_count(a.samples, a.n, a.w, 32), 1, 8);
    if (a.kind == 1) launch_lt_act<W, 1>(a, Wl, b, grid, st);
    else if (a.kind == 3) launch_lt_act<W, 3>(a, Wl, b, grid, st);
    else launch_lt_act<W, 0>(a, Wl, b, grid, st);
}

hipError_t launch_linear_tail_w(const PostArgs& a, const float* Wl, const float* b, hipStream_t st) {
    if (a.samples <= 0) return hipSuccess;
    switch (a.w) {
        case 16: launch_lt<16>(a, Wl, b, st); break;
        case 20: launch_lt<20>(a, Wl, b, st); break;
        case 24: launch_lt<24>(a, Wl, b, st); break;
        case 32: launch_lt<32>(a, Wl, b, st); break;
        case 40: launch_lt<40>(a, Wl, b, st); break;
        default: launch_lt<48>(a, Wl, b, st); break;
    }
    return hipGetLastError();
}

template <int W, int KIND, int ACT>
static void launch_layt_fqn(const LayerTailArgs& a, int int_epi, unsigned grid, hipStream_t st) {
    if (a.p.fq_next.on == 1)
        hipLaunchKernelGGL((k_layer_tail_w<W, KIND, ACT, 1>), dim3(grid), dim3(256), 0, st, a, int_epi);
    else
        hipLaunchKernelGGL((k_layer_tail_w<W, KIND, ACT, 0>), dim3(grid), dim3(256), 0, st, a, int_epi);
}

template <int W, int KIND>
static void launch_layt_act(const LayerTailArgs& a, int int_epi, unsigned grid, hipStream_t st) {
    if (a.p.act == RT_ACT_GELU) launch_layt_fqn<W, KIND, RT_ACT_GELU>(a, int_epi, grid, st);
    else launch_layt_fqn<W, KIND, RT_ACT_RELU>(a, int_epi, grid, st);
}

template <int W>
static void launch_layt(const LayerTailArgs& a, hipStream_t st) {
    const unsigned grid = grid_for(tile_count(a.p.samples, a.p.n, a.p.w, 32), 1, 8);
    const int int_epi = a.zpA != 0 || a.zpW;
    if (a.p.kind == 1) launch_layt_act<W, 1>(a, int_epi, grid, st);
    else if (a.p.kind == 3) launch_layt_act<W, 3>(a, int_epi, grid, st);
    else launch_layt_act<W, 0>(a, int_epi, grid, st);
}

hipError_t launch_layer_tail_w(const LayerTailArgs& a, hipStream_t st) {
    if (a.p.samples <= 0) return hipSuccess;
    switch (a.p.w) {
        case 16: launch_layt<16>(a, st); break;
        case 20: launch_layt<20>(a, st); break;
        case 24: launch_layt<24>(a, st); break;
        case 32: launch_layt<32>(a, st); break;
        case 40: launch_layt<40>(a, st); break;
        default: launch_layt<48>(a, st); break;
    }
    return hipGetLastError();
}

template <int W, int ACT>
static void launch_pt_fq(const ProjArgs& a, unsigned grid, hipStream_t st) {
    if (a.fq_q.on == 1) hipLaunchKernelGGL((k_proj_tail_w<W, ACT, 1>), dim3(grid), dim3(256), 0, st, a);
    else if (a.fq_q.on == 3) hipLaunchKernelGGL((k_proj_tail_w<W, ACT, 3>), dim3(grid), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((k_proj_tail_w<W, ACT, 0>), dim3(grid), dim3(256), 0, st, a);
}

template <int W>
static void launch_pt(const ProjArgs& a, hipStream_t st) {
    const unsigned grid = grid_for(tile_count(a.samples, a.n, a.w, 32), 1, 8);
    if (a.act == RT_ACT_GELU) launch_pt_fq<W, RT_ACT_GELU>(a, grid, st);
    else launch_pt_fq<W, RT_ACT_RELU>(a, grid, st);
}

hipError_t launch_proj_tail_w(const ProjArgs& a, hipStream_t st) {
    if (a.samples <= 0) return hipSuccess;
    switch (a.w) {
        case 16: launch_pt<16>(a, st); break;
        case 20: launch_pt<20>(a, st); break;
        case 24: launch_pt<24>(a, st); break;
        case 32: launch_pt<32>(a, st); break;
        case 40: launch_pt<40>(a, st); break;
        default: launch_pt<48>(a, st); break;
    }
    return hipGetLastError();
}

}  // namespace nfq
