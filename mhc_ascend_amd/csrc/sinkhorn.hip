// Batched Sinkhorn-Knopp forward / exact backward on [batch, n, n] fp32.
//
// Replaces sinkhorn_knopp_forward (sinkhorn_knopp.cpp:739, v3 path 625-665)
// and sinkhorn_knopp_backward (1904, N4 path 1608-1814).  One matrix per
// group of pow2ceil(n) lanes, one row per lane, all iterations in registers;
// column sums are lane-group butterflies.  The backward keeps the forward
// history (post-row-step rows and row sums) in registers and applies the
// exact adjoint (the reference's row step is approximate,
// sinkhorn_knopp.cpp:1773-1795).  Small batches at n = 3..8 run one element
// per lane of a 16-lane DPP row or a wave instead (SkEl in mhc_device.h), 9 <= n
// <= 32 a matrix per wave or workgroup (skw16, skb); n up to 64 (and adjoints
// of more than 32 iterations) the masked wide kernels (skw_*), whose backward
// recomputes the forward state per iteration instead of keeping a history.
#include "mhc_device.h"
#include "mhc_internal.h"

namespace mhc {

template <int N>
__device__ __forceinline__ void load_row(const float* p, float (&a)[N]) {
    if constexpr (N == 4) {
        const float4 q = *reinterpret_cast<const float4*>(p);
        a[0] = q.x; a[1] = q.y; a[2] = q.z; a[3] = q.w;
    } else {
#pragma unroll
        for (int c = 0; c < N; ++c) a[c] = p[c];
    }
}

template <int N>
__device__ __forceinline__ void store_row(float* p, const float (&a)[N]) {
    if constexpr (N == 4) {
        *reinterpret_cast<float4*>(p) = make_float4(a[0], a[1], a[2], a[3]);
    } else {
#pragma unroll
        for (int c = 0; c < N; ++c) p[c] = a[c];
    }
}

template <int N>
__global__ __launch_bounds__(256) void sinkhorn_fwd_kernel(const float* __restrict__ inp, float* __restrict__ out,
                                                           int64_t batch, int iters, float eps) {
    constexpr int G = pow2ceil(N);
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t m = gid / G;
    const int r = (int)(gid % G);
    const bool ok = (m < batch) && (r < N);
    float a[N];
    if (ok) {
        load_row<N>(inp + m * N * N + r * N, a);
    } else {
#pragma unroll
        for (int c = 0; c < N; ++c) a[c] = 0.f;
    }
    sk_forward<N>(a, iters, eps, ok);
    if (ok) store_row<N>(out + m * N * N + r * N, a);
}

template <int N>
__global__ __launch_bounds__(256) void sinkhorn_bwd_kernel(const float* __restrict__ grad_out,
                                                           const float* __restrict__ inp,
                                                           float* __restrict__ grad_inp, int64_t batch, int iters,
                                                           float eps) {
    constexpr int G = pow2ceil(N);
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t m = gid / G;
    const int r = (int)(gid % G);
    const bool ok = (m < batch) && (r < N);
    float x0[N], g[N];
    if (ok) {
        load_row<N>(inp + m * N * N + r * N, x0);
        load_row<N>(grad_out + m * N * N + r * N, g);
    } else {
#pragma unroll
        for (int c = 0; c < N; ++c) { x0[c] = 0.f; g[c] = 0.f; }
    }
    sk_backward<N>(g, x0, iters, eps, ok);
    if (ok) store_row<N>(grad_inp + m * N * N + r * N, g);
}

// n = 3..8: one matrix per S x S lanes, one element per lane (SkEl).  The
// chain per matrix is about S times shorter than with one row per lane but
// issues more instructions in total, so it is used for batches that leave the
// chip latency-bound; large batches (throughput-bound) keep one row per lane,
// except where that form's adjoint recomputes its history (n = 5..8 past
// SkHist's iterations: O(iters^2) steps).  n = 5..8, whose matrix takes a whole
// wave: 8.9 us for 47 at 2048 matrices, 20 iterations, backward; forward 9.5 for
// 8.2 at 8192.
constexpr int64_t sk_el_max_batch(int n) { return n <= 4 ? 16384 : 4096; }
template <int S>
__global__ __launch_bounds__(256) void sinkhorn_el_fwd_kernel(const float* __restrict__ inp, float* __restrict__ out,
                                                              int n, int64_t batch, int iters, float eps) {
    constexpr int L = SkEl<S>::kLanes;
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t m = gid / L;
    const int r = (int)(gid % L) / S, c = (int)(gid % S);
    const bool on = m < batch && r < n && c < n;
    const int64_t at = m * n * n + r * n + c;
    float a = on ? inp[at] : 0.f;
    SkEl<S>::forward(a, iters, SkEl<S>::pad_eps(r, n, eps), SkEl<S>::pad_eps(c, n, eps));
    if (on) out[at] = a;
}

template <int S>
__global__ __launch_bounds__(256) void sinkhorn_el_bwd_kernel(const float* __restrict__ grad_out,
                                                              const float* __restrict__ inp,
                                                              float* __restrict__ grad_inp, int n, int64_t batch,
                                                              int iters, float eps) {
    constexpr int L = SkEl<S>::kLanes;
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t m = gid / L;
    const int r = (int)(gid % L) / S, c = (int)(gid % S);
    const bool on = m < batch && r < n && c < n;
    const int64_t at = m * n * n + r * n + c;
    float g = on ? grad_out[at] : 0.f;
    const float x0 = on ? inp[at] : 0.f;
    SkEl<S>::backward(g, x0, iters, SkEl<S>::pad_eps(r, n, eps), SkEl<S>::pad_eps(c, n, eps), on);
    if (on) grad_inp[at] = g;
}

// 8 < n <= 64: one matrix per group of NM = pow2ceil(n) lanes (16, 32 or
// 64), one row per lane, n taken at run time with the padded columns masked.
template <int NM>
__global__ __launch_bounds__(256) void sinkhorn_wide_fwd_kernel(const float* __restrict__ inp,
                                                                float* __restrict__ out, int n, int64_t batch,
                                                                int iters, float eps) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t m = gid / NM;
    const int r = (int)(gid % NM);
    const bool ok = (m < batch) && (r < n);
    const float* row = inp + (m * n + r) * n;
    float a[NM];
#pragma unroll
    for (int c = 0; c < NM; ++c) a[c] = (ok && c < n) ? row[c] : 0.f;
    skw_forward<NM>(a, n, iters, eps, ok);
    if (ok) {
        float* o = out + (m * n + r) * n;
#pragma unroll
        for (int c = 0; c < NM; ++c) {
            if (c < n) o[c] = a[c];
        }
    }
}

template <int NM>
__global__ __launch_bounds__(256) void sinkhorn_wide_bwd_kernel(const float* __restrict__ grad_out,
                                                                const float* __restrict__ inp,
                                                                float* __restrict__ grad_inp, int n, int64_t batch,
                                                                int iters, float eps) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t m = gid / NM;
    const int r = (int)(gid % NM);
    const bool ok = (m < batch) && (r < n);
    const int64_t off = (m * n + r) * n;
    float x0[NM], g[NM];
#pragma unroll
    for (int c = 0; c < NM; ++c) {
        x0[c] = (ok && c < n) ? inp[off + c] : 0.f;
        g[c] = (ok && c < n) ? grad_out[off + c] : 0.f;
    }
    skw_backward<NM>(g, x0, n, iters, eps, ok);
    if (ok) {
#pragma unroll
        for (int c = 0; c < NM; ++c) {
            if (c < n) grad_inp[off + c] = g[c];
        }
    }
}

// 9 <= n <= 16: one matrix per wave, four elements per lane (skw16); 17 <= n
// <= 32: one matrix per 256-lane workgroup (skb).  The row-per-lane kernels
// above walk 16 or 32 columns of lane-group reductions per iteration, and
// their adjoint recomputes each iteration's state; these keep it in registers
// (up to kTMax = 32 iterations).
__global__ __launch_bounds__(256) void sinkhorn_w16_kernel(const float* __restrict__ grad_out,
                                                           const float* __restrict__ inp, float* __restrict__ out,
                                                           int n, int64_t batch, int iters, float eps) {
    constexpr int V = skw16::kV;
    const int64_t m = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    const int i = skw16::row(), c0 = skw16::col0();
    const int64_t at = (m * n + i) * n + c0;
    bool on[V];
    float a[V], g[V];
#pragma unroll
    for (int k = 0; k < V; ++k) {
        on[k] = m < batch && i < n && c0 + k < n;
        a[k] = on[k] ? inp[at + k] : 0.f;
        g[k] = on[k] && grad_out ? grad_out[at + k] : 0.f;
    }
    if (grad_out) {  // the same for the whole grid
        skw16::backward_n(g, a, n, iters, eps);
    } else {
        skw16::forward_n(a, n, iters, eps);
    }
#pragma unroll
    for (int k = 0; k < V; ++k) {
        if (on[k]) out[at + k] = grad_out ? g[k] : a[k];
    }
}

__global__ __launch_bounds__(skb::kThreads) void sinkhorn_b32_kernel(const float* __restrict__ grad_out,
                                                                     const float* __restrict__ inp,
                                                                     float* __restrict__ out, int n, int iters,
                                                                     float eps) {
    constexpr int V = skb::kV;
    __shared__ float part[skb::kPartFloats];
    __shared__ float hc[skb::kHistFloats];
    const int64_t m = blockIdx.x;
    const int i = skb::row(), c0 = skb::col0();
    const int64_t at = (m * n + i) * n + c0;
    bool on[V];
    float a[V], g[V];
#pragma unroll
    for (int k = 0; k < V; ++k) {
        on[k] = i < n && c0 + k < n;
        a[k] = on[k] ? inp[at + k] : 0.f;
        g[k] = on[k] && grad_out ? grad_out[at + k] : 0.f;
    }
    if (grad_out) {  // the same for the whole grid
        skb::backward_n(g, a, n, iters, eps, part, hc);
    } else {
        skb::forward_n(a, n, iters, eps, part);
    }
#pragma unroll
    for (int k = 0; k < V; ++k) {
        if (on[k]) out[at + k] = grad_out ? g[k] : a[k];
    }
}

// Both directions of 9 <= n <= 32 (grad_out null: forward); false: the shape,
// the batch or the iteration count stays with the row-per-lane kernels.
//
// A matrix per wave or workgroup has the short chain, the row-per-lane kernels
// the fewer instructions a matrix: past the batch that fills the chip they are
// faster forward (20 iterations, us, tiled / row per lane: n = 9 9.8 / 11.5 at
// 2048, 33 / 14 at 8192; n = 16 10.5 / 20 at 2048, 34 / 28 at 8192; n = 17 11 / 24 at
// 256, 44 / 27 at 2048; n = 32 47 / 51 at 2048, 170 / 96 at 8192).  Their adjoint
// recomputes the state, iters^2 steps, so backward the line is the batch at few
// iterations only (n = 9 at 131,072: 20 iterations 1086 / 1371, 10 611 / 394; n = 32
// 5234 / 11,018, 3096 / 3221; at 2048 and 10 iterations 12 / 35 and 49 / 128).
static bool sinkhorn_tiled(int n, int64_t batch, int iters, bool bwd) {
    if (n <= 8 || n > skb::kN || batch > 0x7fffffff) return false;
    const bool wave = n <= skw16::kN;
    if (!bwd) return batch <= (wave ? 256 : 48) * (int64_t)n;
    if (iters > (wave ? skw16::kTMax : skb::kTMax)) return false;
    const int64_t steps = (int64_t)n * iters;
    return steps >= (wave ? 170 : 300) || batch <= (wave ? 64 : 16) * steps;
}

static bool launch_sinkhorn_tiled(int n, const float* grad_out, const float* inp, float* out, int64_t batch, int iters,
                                  float eps, hipStream_t s) {
    if (!sinkhorn_tiled(n, batch, iters, grad_out != nullptr)) return false;
    if (n <= skw16::kN) {
        MHC_LAUNCH_GGL(sinkhorn_w16_kernel, dim3((unsigned)((batch + 3) / 4)), dim3(256), 0, s, grad_out, inp, out, n,
                       batch, iters, eps);
    } else {
        MHC_LAUNCH_GGL(sinkhorn_b32_kernel, dim3((unsigned)batch), dim3(skb::kThreads), 0, s, grad_out, inp, out, n,
                       iters, eps);
    }
    return true;
}

#define MHC_SK_WIDE(n, ...)                                                   \
    if (n <= 16) {                                                            \
        constexpr int NM_ = 16; __VA_ARGS__;                                  \
    } else if (n <= 32) {                                                     \
        constexpr int NM_ = 32; __VA_ARGS__;                                  \
    } else if (n <= 64) {                                                     \
        constexpr int NM_ = 64; __VA_ARGS__;                                  \
    } else {                                                                  \
        return hipErrorInvalidValue;                                          \
    }

#define MHC_SK_DISPATCH(n, ...)                                   \
    switch (n) {                                                  \
        case 1: { constexpr int N_ = 1; __VA_ARGS__; break; }     \
        case 2: { constexpr int N_ = 2; __VA_ARGS__; break; }     \
        case 3: { constexpr int N_ = 3; __VA_ARGS__; break; }     \
        case 4: { constexpr int N_ = 4; __VA_ARGS__; break; }     \
        case 5: { constexpr int N_ = 5; __VA_ARGS__; break; }     \
        case 6: { constexpr int N_ = 6; __VA_ARGS__; break; }     \
        case 7: { constexpr int N_ = 7; __VA_ARGS__; break; }     \
        case 8: { constexpr int N_ = 8; __VA_ARGS__; break; }     \
        default: return hipErrorInvalidValue;                     \
    }

hipError_t launch_sinkhorn_fwd(int n, const float* inp, float* out, int64_t batch, int iters, float eps,
                               hipStream_t s) {
    if (batch == 0) return hipSuccess;
    const int G = pow2ceil(n);
    const int64_t threads = batch * G;
    const unsigned blocks = (unsigned)((threads + 255) / 256);
    const int tok = timing_begin("sinkhorn_fwd", s);
    if (n >= 3 && n <= 8 && batch < sk_el_max_batch(n)) {
        if (sk_el_size(n) == 4) {
            MHC_LAUNCH_GGL(sinkhorn_el_fwd_kernel<4>, dim3((unsigned)((batch * 16 + 255) / 256)), dim3(256), 0, s, inp,
                           out, n, batch, iters, eps);
        } else {
            MHC_LAUNCH_GGL(sinkhorn_el_fwd_kernel<8>, dim3((unsigned)((batch + 3) / 4)), dim3(256), 0, s, inp, out, n,
                           batch, iters, eps);
        }
    } else if (launch_sinkhorn_tiled(n, nullptr, inp, out, batch, iters, eps, s)) {
    } else if (n > 8) {
        MHC_SK_WIDE(n, MHC_LAUNCH_GGL((sinkhorn_wide_fwd_kernel<NM_>), dim3(blocks), dim3(256), 0, s, inp, out, n,
                                          batch, iters, eps));
    } else {
        MHC_SK_DISPATCH(n, MHC_LAUNCH_GGL((sinkhorn_fwd_kernel<N_>), dim3(blocks), dim3(256), 0, s, inp, out,
                                              batch, iters, eps));
    }
    timing_end(tok, s);
    return hipGetLastError();
}

hipError_t launch_sinkhorn_bwd(int n, const float* grad_out, const float* inp, float* grad_inp, int64_t batch,
                               int iters, float eps, hipStream_t s) {
    if (batch == 0) return hipSuccess;
    const int G = pow2ceil(n);
    const int64_t threads = batch * G;
    const unsigned blocks = (unsigned)((threads + 255) / 256);
    const int tok = timing_begin("sinkhorn_bwd", s);
    const bool recompute = n > 4 && n <= 8 && iters > SkHist<8>::TMAX;
    if (n >= 3 && n <= 8 && (batch < sk_el_max_batch(n) || recompute)) {
        if (sk_el_size(n) == 4) {
            MHC_LAUNCH_GGL(sinkhorn_el_bwd_kernel<4>, dim3((unsigned)((batch * 16 + 255) / 256)), dim3(256), 0, s,
                           grad_out, inp, grad_inp, n, batch, iters, eps);
        } else {
            MHC_LAUNCH_GGL(sinkhorn_el_bwd_kernel<8>, dim3((unsigned)((batch + 3) / 4)), dim3(256), 0, s, grad_out,
                           inp, grad_inp, n, batch, iters, eps);
        }
    } else if (launch_sinkhorn_tiled(n, grad_out, inp, grad_inp, batch, iters, eps, s)) {
    } else if (n > 8) {
        MHC_SK_WIDE(n, MHC_LAUNCH_GGL((sinkhorn_wide_bwd_kernel<NM_>), dim3(blocks), dim3(256), 0, s, grad_out,
                                          inp, grad_inp, n, batch, iters, eps));
    } else {
        MHC_SK_DISPATCH(n, MHC_LAUNCH_GGL((sinkhorn_bwd_kernel<N_>), dim3(blocks), dim3(256), 0, s, grad_out,
                                              inp, grad_inp, batch, iters, eps));
    }
    timing_end(tok, s);
    return hipGetLastError();
}

}  // namespace mhc
