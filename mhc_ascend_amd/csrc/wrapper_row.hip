// MHCResidualWrapper, run-time n (2..32): the forward row pass, and the
// dynamic-H backward's row sums where the H_res rows of dP vanish
// (wrap_res_grad_vanishes in abi.hip).
//
// Per token, with h_j = h_pre_j, cm_j the column means of M and hs the mean of
// h_post (wrapper_gen.hip):
//   forward   out = hs (xa / rms) w + sum_j cm_j X_j,  xa = sum_j h_j X_j
//   backward  ss = sum xa^2, gwx = sum w G xa, v_j = sum w G X_j,
//             z_j = sum xa X_j
// X_0 = r, X_1 = b and the others are r m_j, m_j = 0.1^(j-1) or 0, rounded to
// the storage dtype.  So with fp32 rows or 'zero' every other stream is a
// multiple of r: its h_j m_j and cm_j m_j join r's coefficients, v_j = m_j v_0,
// z_j = m_j z_0, and the work per element does not depend on n.  With bf16
// 'decay' xa and the mean form X_2..X_5 as they are rounded; from stream 6 on
// the rounding (2^-9 of 1e-5 r) is below fp32's and they join r as well.  The
// sums v_j and z_j form every stream's.
#include "mhc_device.h"
#include "mhc_internal.h"

namespace mhc {

namespace {

constexpr int kExactStreams = 4;  // X_2..X_5 in xa and the mean (bf16 'decay')

// lane j's coefficients of a token and the wave's folded ones (every lane of
// the wave, n <= 32)
struct RowCoef {
    float hl, cl;  // h_pre_j, cm_j of lane j (0 past n)
    float wl;      // d r weight of stream j
    float hs;
    float cr, sr;  // r's coefficient in xa and in the mean, with the streams that join it
    float h1, c1;
    float hx[kExactStreams], cx[kExactStreams];
};

__device__ __forceinline__ float rlane(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

template <int NE>
__device__ __forceinline__ RowCoef row_coefs(const float* __restrict__ cf, int n, bool decay) {
    const int lane = threadIdx.x & (kWave - 1);
    const bool on = lane < n;
    const float inv_n = 1.f / (float)n;
    const int l = on ? lane : 0;
    RowCoef k;
    k.hl = cf[l];
    float hp = cf[n + l];
    float sc = 0.f;
    const float* m = cf + 2 * n + l;
    int i = 0;
    for (; i + 4 <= n; i += 4) {
        const float a = m[i * n], b = m[(i + 1) * n], c = m[(i + 2) * n], d = m[(i + 3) * n];
        sc += (a + b) + (c + d);
    }
    for (; i < n; ++i) sc += m[i * n];
    k.cl = on ? sc * inv_n : 0.f;
    k.hl = on ? k.hl : 0.f;
    hp = on ? hp : 0.f;
    const float mj = decay ? kWrapMult[l] : 0.f;
    k.wl = lane == 0 ? 1.f : (lane == 1 ? 0.f : mj);
    const float fl = lane >= 2 && lane < 2 + NE ? 0.f : k.wl;
    k.hs = group_sum<kWave>(hp) * inv_n;
    k.cr = group_sum<kWave>(k.hl * fl);
    k.sr = group_sum<kWave>(k.cl * fl);
    k.h1 = rlane(k.hl, 1);
    k.c1 = rlane(k.cl, 1);
#pragma unroll
    for (int j = 0; j < kExactStreams; ++j) {
        k.hx[j] = j < NE ? rlane(k.hl, 2 + j) : 0.f;
        k.cx[j] = j < NE ? rlane(k.cl, 2 + j) : 0.f;
    }
    return k;
}

// four channels of a row as loaded
template <typename TX>
struct Raw4 {
    uint32_t w[sizeof(TX)];
    __device__ __forceinline__ void load(const TX* p) {
        if constexpr (sizeof(TX) == 2) {
            const uint2 q = ld8_nt(p);
            w[0] = q.x; w[1] = q.y;
        } else {
            const uint4 q = ld16_nt(p);
            w[0] = q.x; w[1] = q.y; w[2] = q.z; w[3] = q.w;
        }
    }
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int i = 0; i < (int)sizeof(TX); ++i) w[i] = 0u;
    }
    __device__ __forceinline__ float get(int e) const {
        if constexpr (sizeof(TX) == 2) {
            return __uint_as_float((e & 1) ? (w[e >> 1] & 0xffff0000u) : (w[e >> 1] << 16));
        } else {
            return __uint_as_float(w[e]);
        }
    }
};

// stream j of two channels, rounded to bf16
__device__ __forceinline__ void xpair(float r0, float r1, int j, float& x0, float& x1) {
    const uint32_t p = pack_bf16x2(r0 * kWrapMult[j], r1 * kWrapMult[j]);
    x0 = __uint_as_float(p << 16);
    x1 = __uint_as_float(p & 0xffff0000u);
}

// xa and (MEAN) the stream mean of four channels
template <int NE, bool MEAN>
__device__ __forceinline__ void row_mix(const RowCoef& k, const float (&r)[4], const float (&b)[4], float (&xa)[4],
                                        float (&mn)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        xa[e] = fmaf(k.cr, r[e], k.h1 * b[e]);
        if constexpr (MEAN) mn[e] = fmaf(k.sr, r[e], k.c1 * b[e]);
    }
#pragma unroll
    for (int j = 0; j < NE; ++j) {
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
            float x0, x1;
            xpair(r[e], r[e + 1], 2 + j, x0, x1);
            xa[e] = fmaf(k.hx[j], x0, xa[e]);
            xa[e + 1] = fmaf(k.hx[j], x1, xa[e + 1]);
            if constexpr (MEAN) {
                mn[e] = fmaf(k.cx[j], x0, mn[e]);
                mn[e + 1] = fmaf(k.cx[j], x1, mn[e + 1]);
            }
        }
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// Forward row pass.  W waves take a token (W = 1: four tokens a workgroup; else
// the whole workgroup), lane t the 4-channel chunks t, t + 64 W, ..: at most
// VPT of them, so w xa and the mean stay in registers over the row sum, the row
// is read once and its streams are formed once.  Bound by its bytes, 4 B read
// and 4 B written per element of bf16 rows.  65,536 x 7168 bf16 'decay':
// 654 us at n = 8 (5.7 TB/s; 1219 as two passes over the row that each formed
// all eight streams), 607-638 at n = 4 (686 with a token per wave, 112 registers
// of packed row and the streams formed twice); fp32 n = 5, 4096 x 1024: 8.8 us
// for 15.1.
// ---------------------------------------------------------------------------
template <typename TX, int NE, int W, int VPT>
__global__ __launch_bounds__(W == 1 ? 256 : 64 * W) void wrow_fwd_kernel(const TX* __restrict__ res,
                                                                       const TX* __restrict__ br,
                                                                       const float* __restrict__ w,
                                                                       const float* __restrict__ coef,
                                                                       int64_t coef_stride, float* __restrict__ out,
                                                                       int64_t B, int C, int n, int decay, float eps) {
    __shared__ float red[W];
    const int wave = (int)wave_uniform(threadIdx.x / kWave);
    const int64_t b = W == 1 ? (int64_t)blockIdx.x * 4 + wave : (int64_t)blockIdx.x;
    if (b >= B) return;
    const int t = W == 1 ? (int)(threadIdx.x & (kWave - 1)) : (int)threadIdx.x;
    const TX* rb = res + b * (int64_t)C;
    const TX* bb = br + b * (int64_t)C;
    const int nq = C / 4;
    Raw4<TX> rr[VPT], bw[VPT];
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const int q = k * 64 * W + t;
        if (q < nq) {
            rr[k].load(rb + q * 4);
            bw[k].load(bb + q * 4);
        } else {
            rr[k].zero();
            bw[k].zero();
        }
    }
    const RowCoef c = row_coefs<NE>(coef + b * coef_stride, n, decay != 0);
    float xw[VPT][4], mn[VPT][4];
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const int q = k * 64 * W + t;
        const float4 wq = *reinterpret_cast<const float4*>(w + (q < nq ? q : 0) * 4);
        float rv[4], bv[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            rv[e] = rr[k].get(e);
            bv[e] = bw[k].get(e);
        }
        row_mix<NE, true>(c, rv, bv, xw[k], mn[k]);
#pragma unroll
        for (int e = 0; e < 4; ++e) ss = fmaf(xw[k][e], xw[k][e], ss);
        xw[k][0] *= wq.x;
        xw[k][1] *= wq.y;
        xw[k][2] *= wq.z;
        xw[k][3] *= wq.w;
        // formed here: left to the scheduler the means move past the row sum,
        // with the streams kept for them (243 VGPRs instead of 77 at 7 chunks)
#pragma unroll
        for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(xw[k][e]), "+v"(mn[k][e]));
    }
    ss = group_sum<kWave>(ss);
    if constexpr (W > 1) {
        if (t % kWave == 0) red[wave] = ss;
        __syncthreads();
        ss = 0.f;
#pragma unroll
        for (int i = 0; i < W; ++i) ss += red[i];
    }
    const float hsi = c.hs / sqrtf(ss / (float)C + eps);
    float* ob = out + b * (int64_t)C;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const int q = k * 64 * W + t;
        if (q >= nq) continue;
        st16_nt(ob + q * 4, make_uint4(__float_as_uint(fmaf(hsi, xw[k][0], mn[k][0])),
                                       __float_as_uint(fmaf(hsi, xw[k][1], mn[k][1])),
                                       __float_as_uint(fmaf(hsi, xw[k][2], mn[k][2])),
                                       __float_as_uint(fmaf(hsi, xw[k][3], mn[k][3]))));
    }
}

// Rows too long for registers (C > 16384): a wave per token reads its row
// twice, the second time through the cache.
template <typename TX, int NE>
__global__ __launch_bounds__(256) void wrow_fwd_long_kernel(const TX* __restrict__ res, const TX* __restrict__ br,
                                                            const float* __restrict__ w,
                                                            const float* __restrict__ coef, int64_t coef_stride,
                                                            float* __restrict__ out, int64_t B, int C, int n,
                                                            int decay, float eps) {
    constexpr int U = 4;
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t b = (int64_t)blockIdx.x * 4 + (int64_t)wave_uniform(threadIdx.x / kWave);
    if (b >= B) return;
    const RowCoef c = row_coefs<NE>(coef + b * coef_stride, n, decay != 0);
    const TX* rb = res + b * (int64_t)C;
    const TX* bb = br + b * (int64_t)C;
    const int nq = C / 4;
    float ss = 0.f, unused[4];
    for (int q0 = 0; q0 < nq; q0 += U * kWave) {
        float rv[U][4], bv[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int q = q0 + u * kWave + lane;
            const int c0 = (q < nq ? q : 0) * 4;
            load_run<TX, 4>(rb + c0, rv[u]);
            load_run<TX, 4>(bb + c0, bv[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (q0 + u * kWave + lane >= nq) continue;
            float xa[4];
            row_mix<NE, false>(c, rv[u], bv[u], xa, unused);
#pragma unroll
            for (int e = 0; e < 4; ++e) ss = fmaf(xa[e], xa[e], ss);
        }
    }
    const float hsi = c.hs / sqrtf(group_sum<kWave>(ss) / (float)C + eps);
    float* ob = out + b * (int64_t)C;
    for (int q0 = 0; q0 < nq; q0 += U * kWave) {
        float rv[U][4], bv[U][4], wv[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int q = q0 + u * kWave + lane;
            const int c0 = (q < nq ? q : 0) * 4;
            load_run_nt<TX, 4>(rb + c0, rv[u]);
            load_run_nt<TX, 4>(bb + c0, bv[u]);
            load_run<float, 4>(w + c0, wv[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int q = q0 + u * kWave + lane;
            if (q >= nq) continue;
            float xa[4], mn[4], o[4];
            row_mix<NE, true>(c, rv[u], bv[u], xa, mn);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = fmaf(hsi, xa[e] * wv[u][e], mn[e]);
            store_run_nt<float, 4>(ob + q * 4, o);
        }
    }
}

// ---------------------------------------------------------------------------
// Backward row sums of a token, one wave each: scal_out[b][n*n + ..] as
// wgen_red_kernel writes it except the n x n dM, which nothing reads when the
// H_res gradients vanish, and its factor record.  NX: streams past the second
// whose v and z are formed (bf16 'decay': n - 2; else 0).  65,536 x
// 7168 bf16 n = 8: 644 us (5.8 TB/s) for 970 with dM's sums and every stream in
// xa, bound by the vector units there; fp32 n = 5, 4096 x 1024: 11.5 us for 18.6.
// ---------------------------------------------------------------------------
template <typename TX, int NX>
__global__ __launch_bounds__(256) void wrow_red_kernel(const float* __restrict__ g, const TX* __restrict__ res,
                                                       const TX* __restrict__ br, const float* __restrict__ w,
                                                       const float* __restrict__ coef, int64_t coef_stride,
                                                       float* __restrict__ scal_out, float* __restrict__ ep_out,
                                                       int64_t B, int C, int n, int decay, float eps) {
    constexpr int NE = NX < kExactStreams ? NX : kExactStreams;
    constexpr int NV = 2 + NX;
    constexpr int U = 4;
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t b = (int64_t)blockIdx.x * 4 + (int64_t)wave_uniform(threadIdx.x / kWave);
    if (b >= B) return;
    const RowCoef c = row_coefs<NE>(coef + b * coef_stride, n, decay != 0);
    float rs[2 + 2 * NV];
#pragma unroll
    for (int q = 0; q < 2 + 2 * NV; ++q) rs[q] = 0.f;
    const float* gb = g + b * (int64_t)C;
    const TX* rb = res + b * (int64_t)C;
    const TX* bb = br + b * (int64_t)C;
    const int nq = C / 4;
    for (int q0 = 0; q0 < nq; q0 += U * kWave) {
        uint4 graw[U], wraw[U];
        Raw4<TX> rr[U], bw[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int q = q0 + u * kWave + lane;
            const int c0 = (q < nq ? q : 0) * 4;
            graw[u] = ld16_nt(gb + c0);
            wraw[u] = *reinterpret_cast<const uint4*>(w + c0);
            rr[u].load(rb + c0);
            bw[u].load(bb + c0);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (q0 + u * kWave + lane >= nq) continue;
            const uint32_t gw[4] = {graw[u].x, graw[u].y, graw[u].z, graw[u].w};
            const uint32_t ww[4] = {wraw[u].x, wraw[u].y, wraw[u].z, wraw[u].w};
            float rv[4], bv[4], xa[4], wg[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                rv[e] = rr[u].get(e);
                bv[e] = bw[u].get(e);
                wg[e] = __uint_as_float(ww[e]) * __uint_as_float(gw[e]);
                xa[e] = fmaf(c.cr, rv[e], c.h1 * bv[e]);
            }
            // xa first, keeping the streams for v and z
            float x[NX > 0 ? NX : 1][4];
#pragma unroll
            for (int j = 0; j < NX; ++j) {
#pragma unroll
                for (int e = 0; e < 4; e += 2) xpair(rv[e], rv[e + 1], 2 + j, x[j][e], x[j][e + 1]);
                if (j < NE) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) xa[e] = fmaf(c.hx[j], x[j][e], xa[e]);
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                rs[0] = fmaf(xa[e], xa[e], rs[0]);
                rs[1] = fmaf(wg[e], xa[e], rs[1]);
                rs[2] = fmaf(wg[e], rv[e], rs[2]);
                rs[3] = fmaf(wg[e], bv[e], rs[3]);
                rs[2 + NV] = fmaf(xa[e], rv[e], rs[2 + NV]);
                rs[3 + NV] = fmaf(xa[e], bv[e], rs[3 + NV]);
#pragma unroll
                for (int j = 0; j < NX; ++j) {
                    rs[4 + j] = fmaf(wg[e], x[j][e], rs[4 + j]);
                    rs[4 + NV + j] = fmaf(xa[e], x[j][e], rs[4 + NV + j]);
                }
            }
        }
    }
    wave_sum<2 + 2 * NV>(rs);
    const float inv = 1.f / sqrtf(rs[0] / (float)C + eps);
    const float gwx = rs[1];
    const float k2 = c.hs * gwx * inv * inv * inv / (float)C;
    const float hsi = c.hs * inv;
    // lane j: dh_pre_act_j and dh_post_act_j
    float v = c.wl * rs[2], z = c.wl * rs[2 + NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        v = lane == j ? rs[2 + j] : v;
        z = lane == j ? rs[2 + NV + j] : z;
    }
    float* so = scal_out + b * (int64_t)(n * n + 2 * n + 2) + n * n;
    if (lane < n) {
        so[lane] = gwx * inv / (float)n;
        so[n + lane] = hsi * v - k2 * z;
    }
    const float b_r = group_sum<kWave>(c.hl * c.wl);
    const float a_r = group_sum<kWave>(c.cl * c.wl);
    if (lane < 2) so[2 * n + lane] = lane == 0 ? inv : k2;
    const float rec[8] = {a_r, b_r * hsi, c.c1, c.h1 * hsi, hsi, -b_r * k2, -c.h1 * k2, b_r};
    float ev = __shfl(c.hl, (lane - 8) & (kWave - 1));  // h_pre_0..7
#pragma unroll
    for (int k = 0; k < 8; ++k) ev = lane == k ? rec[k] : ev;
    if (lane < kWgEp) ep_out[b * kWgEp + lane] = ev;
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
hipError_t launch_wrow_fwd(int dt, int n, bool decay, const void* res, const void* br, const float* w,
                           const float* coef, int64_t coef_stride, float* out, int64_t B, int64_t C, float eps,
                           hipStream_t s) {
    if (B == 0) return hipSuccess;
    if (!wgen_supported(n, C)) return hipErrorInvalidValue;
    const int Ci = (int)C, dec = decay ? 1 : 0;
    const int64_t nq = C / 4;
    const bool exact = dt == kBF16 && decay && n > 2;
    // waves of a token: one to 2048 channels, four to 8192, eight to 16384
    const int W = nq <= 512 ? 1 : (nq <= 2048 ? 4 : (nq <= 4096 ? 8 : 0));
    const int64_t blocks = W <= 1 ? (B + 3) / 4 : B;
    if (blocks > 0x7fffffff) return hipErrorInvalidValue;
    const dim3 grid((unsigned)blocks);
    const int vpt = W ? (int)((nq + 64 * W - 1) / (64 * W)) : 0;
    const int tok = timing_begin("wrap_fwd", s);
#define MHC_WRF_(TX_, NE_, W_, V_)                                                                                    \
    MHC_LAUNCH_GGL((wrow_fwd_kernel<TX_, NE_, W_, V_>), grid, dim3(W_ == 1 ? 256 : 64 * W_), 0, s, (const TX_*)res,   \
                   (const TX_*)br, w, coef, coef_stride, out, B, Ci, n, dec, eps)
#define MHC_WRF(TX_, NE_)                                                                                             \
    if (W == 1) {                                                                                                     \
        if (vpt <= 1) { MHC_WRF_(TX_, NE_, 1, 1); }                                                                   \
        else if (vpt == 2) { MHC_WRF_(TX_, NE_, 1, 2); }                                                              \
        else if (vpt <= 4) { MHC_WRF_(TX_, NE_, 1, 4); }                                                              \
        else if (vpt <= 6) { MHC_WRF_(TX_, NE_, 1, 6); }                                                              \
        else { MHC_WRF_(TX_, NE_, 1, 8); }                                                                            \
    } else if (W == 4) {                                                                                              \
        if (vpt <= 3) { MHC_WRF_(TX_, NE_, 4, 3); }                                                                   \
        else if (vpt == 4) { MHC_WRF_(TX_, NE_, 4, 4); }                                                              \
        else if (vpt == 5) { MHC_WRF_(TX_, NE_, 4, 5); }                                                              \
        else if (vpt == 6) { MHC_WRF_(TX_, NE_, 4, 6); }                                                              \
        else if (vpt == 7) { MHC_WRF_(TX_, NE_, 4, 7); }                                                              \
        else { MHC_WRF_(TX_, NE_, 4, 8); }                                                                            \
    } else if (W == 8) {                                                                                              \
        if (vpt <= 6) { MHC_WRF_(TX_, NE_, 8, 6); }                                                                   \
        else { MHC_WRF_(TX_, NE_, 8, 8); }                                                                            \
    } else {                                                                                                          \
        MHC_LAUNCH_GGL((wrow_fwd_long_kernel<TX_, NE_>), grid, dim3(256), 0, s, (const TX_*)res, (const TX_*)br, w,   \
                       coef, coef_stride, out, B, Ci, n, dec, eps);                                                   \
    }
    // NE counts streams that exist: an absent one would turn an infinite r into
    // 0 x inf
    if (exact && n >= 6) {
        MHC_WRF(bf16_t, kExactStreams)
    } else if (exact && n == 5) {
        MHC_WRF(bf16_t, 3)
    } else if (exact && n == 4) {
        MHC_WRF(bf16_t, 2)
    } else if (exact) {
        MHC_WRF(bf16_t, 1)
    } else if (dt == kBF16) {
        MHC_WRF(bf16_t, 0)
    } else {
        MHC_WRF(float, 0)
    }
#undef MHC_WRF
#undef MHC_WRF_
    timing_end(tok, s);
    return hipGetLastError();
}

// bf16 'decay' past n = 8 would keep more sums than wgen_red_kernel's registers
// and gain nothing
bool wrow_red_ok(int dt, int n, bool decay, int64_t C) {
    return wgen_supported(n, C) && (dt != kBF16 || !decay || n <= 8);
}

hipError_t launch_wrow_red(int dt, int n, bool decay, const float* g, const void* res, const void* br, const float* w,
                           const float* coef, int64_t coef_stride, float* scal_out, float* ep_out, int64_t B,
                           int64_t C, float eps, hipStream_t s) {
    if (B == 0) return hipSuccess;
    if (!wrow_red_ok(dt, n, decay, C)) return hipErrorInvalidValue;
    const int64_t blocks = (B + 3) / 4;
    if (blocks > 0x7fffffff) return hipErrorInvalidValue;
    const int Ci = (int)C, dec = decay ? 1 : 0;
    const int tok = timing_begin("wrap_bwd_red", s);
#define MHC_WRR(TX_, NX_)                                                                                            \
    MHC_LAUNCH_GGL((wrow_red_kernel<TX_, NX_>), dim3((unsigned)blocks), dim3(256), 0, s, g, (const TX_*)res,         \
                   (const TX_*)br, w, coef, coef_stride, scal_out, ep_out, B, Ci, n, dec, eps)
    if (dt != kBF16) {
        MHC_WRR(float, 0);
    } else {
        switch (decay ? n - 2 : 0) {
            case 0: MHC_WRR(bf16_t, 0); break;
            case 1: MHC_WRR(bf16_t, 1); break;
            case 2: MHC_WRR(bf16_t, 2); break;
            case 3: MHC_WRR(bf16_t, 3); break;
            case 4: MHC_WRR(bf16_t, 4); break;
            case 5: MHC_WRR(bf16_t, 5); break;
            default: MHC_WRR(bf16_t, 6); break;
        }
    }
#undef MHC_WRR
    timing_end(tok, s);
    return hipGetLastError();
}

}  // namespace mhc
