// MHCResidualWrapper, dynamic-H backward past the row sums, where the H_res
// rows of dP vanish (wrap_res_grad_vanishes in abi.hip): d r, d b, the dw
// partials and the dPhi partials of the 2n pre / post rows in one pass over
// G, r and b, and the parameter gradients' sums in one launch.
//
// Per token, with the factor record of wgen_red_kernel and w_j the d r weight
// of stream j (1, 0, 0.1, 0.01, .. or 0 past stream 1 in 'zero' mode):
//   d r = A_r G + B_r gxa + s sum_j w_j X_j + dP . Phi_r,  Phi_r = sum_j w_j Phi_j
//   d b = A_b G + B_b gxa + s b + dP . Phi_1
//   dPhi_j = sum_tokens dP X_j
// fp32 rows and 'zero' need two products for dPhi, dP^T r and dP^T b: the
// streams past the second are w_j r to fp32 rounding, so the sum kernel writes
// w_j times the first one's total.  bf16 'decay' rows keep one per stream (the
// rounding of X_j is 2^-9 of it).  In the sums over streams a rounding is left
// out only where it is under fp32's 2^-24 of r: from stream 7 on in xa (2^-9 w_j),
// from stream 4 on in s sum_j w_j X_j (2^-9 w_j^2).
//
// The stage structure is wrap_proj_bwd_kernel's (wrapper.hip): 8 waves x 16
// channels, 32-token stages of r, b and G in LDS, fetched three stages ahead
// into three register sets through buffer resources (two where three do not fit:
// fp32 rows, n > 16).  Rows of dP: 16 MI, split h + m + l (bf16,
// all 24 bits) token-major and h + m output-major.
//   dPhi: D[row][channel] += dP_h X + dP_m X (+ dP_h X_m with fp32 rows)
//   dx:   D[channel][token] += the six products of Phi's and dP's h, m, l down
//         to 2^-24, so as exact as fp32 products; with 16 rows two of them
//         share an MFMA's 32 k: [Phi_h | Phi_m] [dP_h | dP_h], [Phi_h | Phi_m]
//         [dP_m | dP_m], [Phi_l | Phi_h] [dP_h | dP_l]
// What bounds it: its byte mix, 8 B read and 4 B written per element of bf16
// rows, one workgroup per CU.  n = 8, 65,536 x 7168 bf16: 1.28 ms (4.4 TB/s)
// where a dPhi pass and a d r / d b pass over the same rows took 1.27 + 1.89;
// n = 16, 4096 x 2048 fp32: 39 us for 905 through stream rows in memory.
#include "mhc_device.h"
#include "mhc_internal.h"
#include "wrapper_plan.h"

namespace mhc {

namespace {

typedef __bf16 vbf16x8_t __attribute__((ext_vector_type(8)));
typedef float vf32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int vu32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ vf32x4_t vmfma(vu32x4_t a, vu32x4_t b, vf32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(vbf16x8_t, a), __builtin_bit_cast(vbf16x8_t, b),
                                                   c, 0, 0, 0);
}

// 8 fp32 -> bf16 parts in operand order
__device__ __forceinline__ void vsplit8(const float (&v)[8], vu32x4_t& hi, vu32x4_t& mid) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        hi[e] = pack_bf16x2(v[2 * e], v[2 * e + 1]);
        mid[e] = pack_bf16x2(v[2 * e] - __uint_as_float(hi[e] << 16),
                             v[2 * e + 1] - __uint_as_float(hi[e] & 0xffff0000u));
    }
}
__device__ __forceinline__ void vsplit8(const float (&v)[8], vu32x4_t& hi, vu32x4_t& mid, vu32x4_t& lo) {
    vsplit8(v, hi, mid);
#pragma unroll
    for (int e = 0; e < 4; ++e)
        lo[e] = pack_bf16x2(v[2 * e] - __uint_as_float(hi[e] << 16) - __uint_as_float(mid[e] << 16),
                            v[2 * e + 1] - __uint_as_float(hi[e] & 0xffff0000u) -
                                __uint_as_float(mid[e] & 0xffff0000u));
}

template <typename TX>
__device__ __forceinline__ void vlds_get4(const char* p, float (&v)[4]) {
    const uint2* q = reinterpret_cast<const uint2*>(p);
    if constexpr (sizeof(TX) == 2) {
        const uint2 w = q[0];
        v[0] = __uint_as_float(w.x << 16); v[1] = __uint_as_float(w.x & 0xffff0000u);
        v[2] = __uint_as_float(w.y << 16); v[3] = __uint_as_float(w.y & 0xffff0000u);
    } else {
        const uint2 a = q[0], b = q[1];
        v[0] = __uint_as_float(a.x); v[1] = __uint_as_float(a.y);
        v[2] = __uint_as_float(b.x); v[3] = __uint_as_float(b.y);
    }
}
template <typename TX>
__device__ __forceinline__ void vlds_put4(char* p, const float (&v)[4]) {
    uint2* q = reinterpret_cast<uint2*>(p);
    if constexpr (sizeof(TX) == 2) {
        q[0] = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
    } else {
        q[0] = make_uint2(__float_as_uint(v[0]), __float_as_uint(v[1]));
        q[1] = make_uint2(__float_as_uint(v[2]), __float_as_uint(v[3]));
    }
}

constexpr int kVbThreads = 512;
constexpr int kVbCols = kVbThreads / 64 * 16;
static_assert(kVbCols == kWbwdCols, "the host's column blocks");
constexpr int kVbEp = kWgEp + 4;  // the record, then s (padded to 16 bytes)

}  // namespace

// Phi_r and Phi_1 of the 2n pre / post rows: out[0][o][c], out[1][o][c].  For
// n > 8, where folding them in every workgroup would read n streams of 2n rows
// once per token tile.
__global__ __launch_bounds__(256) void wbwd_fold_phi_kernel(const float* __restrict__ pre, const float* __restrict__ post,
                                                            int n, int C, int decay, float* __restrict__ out) {
    const int64_t total = (int64_t)2 * n * C;
    const int64_t K = (int64_t)n * C;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int o = (int)(i / C);
        const int c = (int)(i - (int64_t)o * C);
        const float* row = (o < n ? pre + (int64_t)o * K : post + (int64_t)(o - n) * K) + c;
        float r = row[0];
        if (decay) {
            double md = 1.0;
            for (int j = 2; j < n; ++j) {
                md *= 0.1;
                r = fmaf((float)md, row[(int64_t)j * C], r);
            }
        }
        out[i] = r;
        out[total + i] = row[C];
    }
}

// NST: streams whose dPhi is formed (2: r and b; else all n, with bf16
// 'decay').  fold: wbwd_fold_phi_kernel's output, or null (n <= 8).
template <typename TX, int NST, int MI>
__global__ __launch_bounds__(kVbThreads) __attribute__((amdgpu_waves_per_eu(2))) void wbwd_kernel(
    const float* __restrict__ g, const TX* __restrict__ res, const TX* __restrict__ br, const float* __restrict__ w,
    const float* __restrict__ ep, const float* __restrict__ dP, int dp_stride, const float* __restrict__ s_tok,
    const float* __restrict__ phi_pre, const float* __restrict__ phi_post, const float* __restrict__ fold, int n,
    int decay, float wsq, TX* __restrict__ dres, TX* __restrict__ dbr, float* __restrict__ dw_part,
    float* __restrict__ dphi_part, int64_t B, int C, int64_t tile) {
    constexpr bool XS = NST > 2;  // rounded streams past the second (n = NST)
    static_assert(!XS || (sizeof(TX) == 2 && NST <= 8 && MI == 1), "bf16 'decay' rows, n = 3..8");
    constexpr int TB = 32;
    constexpr int NT = kVbThreads;
    constexpr int CB = kVbCols;
    constexpr int EPV = 16 / sizeof(TX);
    constexpr int VPR = CB / EPV;
    constexpr int RPP = NT / VPR;
    constexpr int PASSES = TB / RPP;
    constexpr int GVPR = CB / 4;
    constexpr int GRPP = NT / GVPR;
    constexpr int GPASSES = TB / GRPP;
    constexpr int PITCH = CB * (int)sizeof(TX) + 8;
    constexpr int GPITCH = CB * 4 + 16;
    constexpr int RW = 16 * MI;                  // rows of dP carried
    constexpr int KB = MI == 1 ? 1 : MI / 2;     // 32-row k blocks of dx
    constexpr int DEPTH = sizeof(TX) == 4 || MI > 2 ? 2 : 3;  // stages ahead
    constexpr int TP = RW + 8;                   // pitch of the token-major copies (bf16)
    constexpr int OP = TB + 8;                   // pitch of the output-major copies
    static_assert(PASSES * RPP == TB && GPASSES * GRPP == TB && (MI == 1 || MI % 2 == 0) && MI <= 4, "stage shape");
    __shared__ __align__(16) char rb_lds[2][TB * PITCH];
    __shared__ __align__(16) char g_lds[TB * GPITCH];
    __shared__ __align__(16) char out_lds[2][TB * PITCH];
    __shared__ __align__(16) bf16_t dt_lds[3][TB * TP];  // h, m, l: [token][row]
    __shared__ __align__(16) bf16_t do_lds[2][RW * OP];  // h, m: [row][token]
    __shared__ __align__(16) float ep_lds[TB][kVbEp];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int lr = lane & 15;
    const int lg = lane >> 4;
    const int rows = 2 * n;
    const int64_t K = (int64_t)n * C;
    const int64_t cb0 = (int64_t)blockIdx.x * CB;
    const int wc0 = wave * 16;
    const bool wave_on = cb0 + wc0 < C;

    const int lrow = tid / VPR;
    const int lvec = tid % VPR;
    const int64_t lcol = cb0 + (int64_t)lvec * EPV;
    const bool lcol_ok = lcol < C;  // C % 8 == 0: whole pieces
    const int grow = tid / GVPR;
    const int gvec = tid % GVPR;
    const int64_t gcol = cb0 + (int64_t)gvec * 4;
    const bool dp_loader = tid < 8 * RW;
    const int dtk = (tid / (4 * MI)) % TB;
    const int dpo = (tid % (4 * MI)) * 4;
    const bool ep_loader = tid < 4 * TB;
    const int etk = (tid >> 2) % TB;
    const int epc = tid & 3;

    // dx A operands at channel wc0 + lr.  MI = 1: row 8 (lg & 1) + e, Phi_h
    // for lg < 2 and Phi_m above (q[0]), Phi_l and Phi_h (q[1]); else per k
    // block row 32 kb + 8 lg + e, h, m, l (q[3 kb ..])
    constexpr int NQ = MI == 1 ? 2 : 3 * KB;
    vu32x4_t qr[NQ], qb[NQ];
    {
        const int64_t c = cb0 + wc0 + lr;
        const bool on = c < C;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            float vr[8], vb[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int o = MI == 1 ? 8 * (lg & 1) + e : 32 * kb + 8 * lg + e;
                float r = 0.f, b = 0.f;
                if (on && o < rows) {
                    if (fold) {
                        r = fold[(int64_t)o * C + c];
                        b = fold[((int64_t)rows + o) * C + c];
                    } else {
                        const float* rowp = (o < n ? phi_pre + (int64_t)o * K : phi_post + (int64_t)(o - n) * K) + c;
                        r = rowp[0];
                        b = rowp[C];
                        if (decay) {
#pragma unroll
                            for (int j = 2; j < 8; ++j) {
                                if (j < n) r = fmaf(kWrapMult[j], rowp[(int64_t)j * C], r);
                            }
                        }
                    }
                }
                vr[e] = r;
                vb[e] = b;
            }
            if constexpr (MI == 1) {
                vu32x4_t h, m, l;
                vsplit8(vr, h, m, l);
                qr[0] = lg < 2 ? h : m;
                qr[1] = lg < 2 ? l : h;
                vsplit8(vb, h, m, l);
                qb[0] = lg < 2 ? h : m;
                qb[1] = lg < 2 ? l : h;
            } else {
                vsplit8(vr, qr[3 * kb], qr[3 * kb + 1], qr[3 * kb + 2]);
                vsplit8(vb, qb[3 * kb], qb[3 * kb + 1], qb[3 * kb + 2]);
            }
        }
    }
    float wv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t c = cb0 + wc0 + 4 * lg + i;
        wv[i] = c < C ? w[c] : 0.f;
    }
    vf32x4_t acc[NST][MI];
#pragma unroll
    for (int j = 0; j < NST; ++j) {
#pragma unroll
        for (int m = 0; m < MI; ++m) acc[j][m] = vf32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    float dwacc[4] = {0.f, 0.f, 0.f, 0.f};

    const int64_t t_begin = (int64_t)blockIdx.y * tile;
    const int64_t t_end = (t_begin + tile < B) ? t_begin + tile : B;
    const int64_t nrows = t_end > t_begin ? t_end - t_begin : 0;
    const int64_t tb0 = nrows > 0 ? t_begin : 0;

    // buffer resources over the tile's rows (under 2 GiB each, six stages of
    // overrun included: wbwd_tiles); rows past t_end read zeros, stores there
    // are dropped
    const uint32_t xrow = (uint32_t)C * (uint32_t)sizeof(TX);
    const buf_rsrc_t rs_r = make_buf_rsrc(res + tb0 * C, (uint32_t)(nrows * xrow));
    const buf_rsrc_t rs_b = make_buf_rsrc(br + tb0 * C, (uint32_t)(nrows * xrow));
    const buf_rsrc_t rs_g = make_buf_rsrc(g + tb0 * C, (uint32_t)(nrows * C * 4));
    const buf_rsrc_t rs_dr = make_buf_rsrc(dres + tb0 * C, (uint32_t)(nrows * xrow));
    const buf_rsrc_t rs_db = make_buf_rsrc(dbr + tb0 * C, (uint32_t)(nrows * xrow));
    const buf_rsrc_t rs_p = make_buf_rsrc(dP + tb0 * dp_stride, (uint32_t)(nrows * dp_stride * 4));
    const buf_rsrc_t rs_e = make_buf_rsrc(ep + tb0 * kWgEp, (uint32_t)(nrows * kWgEp * 4));
    const buf_rsrc_t rs_s = make_buf_rsrc(s_tok + tb0, (uint32_t)(nrows * 4));
    const uint32_t xo = lcol_ok ? (uint32_t)lrow * xrow + (uint32_t)(lcol * (int64_t)sizeof(TX)) : kBufOff;
    const uint32_t go = gcol < C ? ((uint32_t)grow * (uint32_t)C + (uint32_t)gcol) * 4u : kBufOff;
    const uint32_t po = dp_loader ? (uint32_t)(dtk * dp_stride + dpo) * 4u : kBufOff;
    const uint32_t eo = ep_loader ? (uint32_t)(etk * kWgEp + 4 * epc) * 4u : kBufOff;
    const uint32_t so = (ep_loader && epc == 3) ? (uint32_t)etk * 4u : kBufOff;

    struct Fetched {
        uint4 v[2][PASSES];
        uint4 gq[GPASSES];
        uint4 e, dp;
        uint32_t s;
    };
    Fetched f0, f1, f2;
    auto fetch = [&](Fetched& f, uint32_t rel) __attribute__((always_inline)) {
        f.dp = buf_ld16<false>(rs_p, po + rel * (uint32_t)dp_stride * 4u, 0u);
        f.e = buf_ld16<false>(rs_e, eo + rel * (uint32_t)(kWgEp * 4), 0u);
        f.s = buf_ld4(rs_s, so + rel * 4u, 0u);
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            const uint32_t off = xo + (rel + p * RPP) * xrow;
            f.v[0][p] = buf_ld16<true>(rs_r, off, 0u);
            f.v[1][p] = buf_ld16<true>(rs_b, off, 0u);
        }
#pragma unroll
        for (int p = 0; p < GPASSES; ++p)
            f.gq[p] = buf_ld16<true>(rs_g, go + (rel + p * GRPP) * (uint32_t)C * 4u, 0u);
    };
    auto commit = [&](const Fetched& f) __attribute__((always_inline)) {
        // (see wrap_proj_bwd_kernel: a use of the small records outside their
        // branches keeps the wait counts exact)
        asm volatile("" ::"v"(f.dp.x), "v"(f.dp.y), "v"(f.dp.z), "v"(f.dp.w), "v"(f.e.x), "v"(f.e.y), "v"(f.e.z),
                     "v"(f.e.w), "v"(f.s));
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            const int row = lrow + p * RPP;
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const uint4 v = f.v[a][p];
                uint2* pw = reinterpret_cast<uint2*>(&rb_lds[a][row * PITCH + lvec * 16]);
                pw[0] = make_uint2(v.x, v.y);
                pw[1] = make_uint2(v.z, v.w);
            }
        }
#pragma unroll
        for (int p = 0; p < GPASSES; ++p)
            *reinterpret_cast<uint4*>(&g_lds[(grow + p * GRPP) * GPITCH + gvec * 16]) = f.gq[p];
        if (dp_loader) {
            const uint32_t dw4[4] = {f.dp.x, f.dp.y, f.dp.z, f.dp.w};
            float rest[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) rest[q] = dpo + q < rows ? __uint_as_float(dw4[q]) : 0.f;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const uint32_t p0 = pack_bf16x2(rest[0], rest[1]), p1 = pack_bf16x2(rest[2], rest[3]);
                *reinterpret_cast<uint2*>(&dt_lds[k][dtk * TP + dpo]) = make_uint2(p0, p1);
                if (k < 2) {
                    do_lds[k][(dpo + 0) * OP + dtk] = (bf16_t)(p0 & 0xffffu);
                    do_lds[k][(dpo + 1) * OP + dtk] = (bf16_t)(p0 >> 16);
                    do_lds[k][(dpo + 2) * OP + dtk] = (bf16_t)(p1 & 0xffffu);
                    do_lds[k][(dpo + 3) * OP + dtk] = (bf16_t)(p1 >> 16);
                }
                rest[0] -= __uint_as_float(p0 << 16);
                rest[1] -= __uint_as_float(p0 & 0xffff0000u);
                rest[2] -= __uint_as_float(p1 << 16);
                rest[3] -= __uint_as_float(p1 & 0xffff0000u);
            }
        }
        if (ep_loader) {
            *reinterpret_cast<uint4*>(&ep_lds[etk][4 * epc]) = f.e;
            if (epc == 3) ep_lds[etk][kWgEp] = __uint_as_float(f.s);
        }
    };
    auto read16 = [&](const bf16_t* p) __attribute__((always_inline)) -> vu32x4_t {
        const uint4 q = *reinterpret_cast<const uint4*>(p);
        return vu32x4_t{q.x, q.y, q.z, q.w};
    };
    auto compute = [&]() __attribute__((always_inline)) {
        if (!wave_on) return;
        const char* rt = rb_lds[0];
        const char* bt = rb_lds[1];
        // dPhi: B operands over tokens 8 lg .. + 7 at channel wc0 + lr
        {
            const int c = wc0 + lr;
            vu32x4_t ah[MI], al[MI];
#pragma unroll
            for (int m = 0; m < MI; ++m) {
                ah[m] = read16(&do_lds[0][(16 * m + lr) * OP + 8 * lg]);
                al[m] = read16(&do_lds[1][(16 * m + lr) * OP + 8 * lg]);
            }
            if constexpr (sizeof(TX) == 2) {
                uint32_t rr[8], bb[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int t = 8 * lg + e;
                    rr[e] = *reinterpret_cast<const uint16_t*>(rt + t * PITCH + c * 2);
                    bb[e] = *reinterpret_cast<const uint16_t*>(bt + t * PITCH + c * 2);
                }
                vu32x4_t x0, x1;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x0[e] = rr[2 * e] | (rr[2 * e + 1] << 16);
                    x1[e] = bb[2 * e] | (bb[2 * e + 1] << 16);
                }
#pragma unroll
                for (int m = 0; m < MI; ++m) {
                    acc[0][m] = vmfma(ah[m], x0, acc[0][m]);
                    acc[1][m] = vmfma(ah[m], x1, acc[1][m]);
                    acc[0][m] = vmfma(al[m], x0, acc[0][m]);
                    acc[1][m] = vmfma(al[m], x1, acc[1][m]);
                }
#pragma unroll
                for (int j = 2; j < NST; ++j) {
                    vu32x4_t x;
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        x[e] = pack_bf16x2(__uint_as_float(rr[2 * e] << 16) * kWrapMult[j],
                                           __uint_as_float(rr[2 * e + 1] << 16) * kWrapMult[j]);
                    acc[j][0] = vmfma(ah[0], x, acc[j][0]);
                    acc[j][0] = vmfma(al[0], x, acc[j][0]);
                }
            } else {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const char* src = j == 0 ? rt : bt;
                    float v[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        v[e] = *reinterpret_cast<const float*>(src + (8 * lg + e) * PITCH + c * 4);
                    vu32x4_t xh, xl;
                    vsplit8(v, xh, xl);
#pragma unroll
                    for (int m = 0; m < MI; ++m) {
                        acc[j][m] = vmfma(ah[m], xh, acc[j][m]);
                        acc[j][m] = vmfma(al[m], xh, acc[j][m]);
                        acc[j][m] = vmfma(ah[m], xl, acc[j][m]);
                    }
                }
            }
        }
        // d r, d b of token 16 tt + lr, channels wc0 + 4 lg .. + 3
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            const int t = 16 * tt + lr;
            vf32x4_t pr = vf32x4_t{0.f, 0.f, 0.f, 0.f}, pb = pr;
            if constexpr (MI == 1) {
                const vu32x4_t bh = read16(&dt_lds[0][t * TP + 8 * (lg & 1)]);
                const vu32x4_t bm = read16(&dt_lds[1][t * TP + 8 * (lg & 1)]);
                const vu32x4_t bl = read16(&dt_lds[lg < 2 ? 0 : 2][t * TP + 8 * (lg & 1)]);
                pr = vmfma(qr[1], bl, pr);
                pb = vmfma(qb[1], bl, pb);
                pr = vmfma(qr[0], bm, pr);
                pb = vmfma(qb[0], bm, pb);
                pr = vmfma(qr[0], bh, pr);
                pb = vmfma(qb[0], bh, pb);
            } else {
#pragma unroll
                for (int kb = 0; kb < KB; ++kb) {
                    // dP parts h, m, l against the Phi parts that reach 2^-24
#pragma unroll
                    for (int k = 2; k >= 0; --k) {
                        const vu32x4_t d = read16(&dt_lds[k][t * TP + 32 * kb + 8 * lg]);
#pragma unroll
                        for (int q = 2 - k; q >= 0; --q) {
                            pr = vmfma(qr[3 * kb + q], d, pr);
                            pb = vmfma(qb[3 * kb + q], d, pb);
                        }
                    }
                }
            }
            const float4 e0 = *reinterpret_cast<const float4*>(&ep_lds[t][0]);
            const float4 e1 = *reinterpret_cast<const float4*>(&ep_lds[t][4]);
            const float4 h0 = *reinterpret_cast<const float4*>(&ep_lds[t][8]);
            const float4 h1 = *reinterpret_cast<const float4*>(&ep_lds[t][12]);
            const float st = ep_lds[t][kWgEp];
            const float a_r = e0.x, brh = e0.y, a_b = e0.z, bbh = e0.w;
            const float hsi = e1.x, kr = e1.y, kb2 = e1.z;
            const float hp[8] = {h0.x, h0.y, h0.z, h0.w, h1.x, h1.y, h1.z, h1.w};
            // xa = cr r + h_1 b (+ the rounded streams): without them every
            // stream of r is a multiple of it (e1.w = sum_j w_j h_j); with them
            // stream 7 joins the multiple (its rounding is 2^-9 1e-6 = 2^-29 of r)
            const float cr = XS ? (NST > 7 ? fmaf(hp[7], kWrapMult[7], hp[0]) : hp[0]) : e1.w;
            const int col = wc0 + 4 * lg;
            const int boff = t * PITCH + col * (int)sizeof(TX);
            float rv[4], bv[4];
            vlds_get4<TX>(rt + boff, rv);
            vlds_get4<TX>(bt + boff, bv);
            const float4 gq = *reinterpret_cast<const float4*>(&g_lds[t * GPITCH + col * 4]);
            const float gv[4] = {gq.x, gq.y, gq.z, gq.w};
            float drv[4], dbv[4], xav[4], sxv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                xav[i] = fmaf(cr, rv[i], hp[1] * bv[i]);
                sxv[i] = rv[i] * wsq;
            }
            if constexpr (XS) {
#pragma unroll
                for (int j = 2; j < (NST < 7 ? NST : 7); ++j) {
#pragma unroll
                    for (int i = 0; i < 4; i += 2) {
                        const uint32_t x2 = pack_bf16x2(rv[i] * kWrapMult[j], rv[i + 1] * kWrapMult[j]);
                        const float x0 = __uint_as_float(x2 << 16), x1 = __uint_as_float(x2 & 0xffff0000u);
                        xav[i] = fmaf(hp[j], x0, xav[i]);
                        xav[i + 1] = fmaf(hp[j], x1, xav[i + 1]);
                        if (j < 4) {  // wsq holds the others as w_j^2 r: 2^-9 w_4^2 < 2^-28
                            sxv[i] = fmaf(kWrapMult[j], x0, sxv[i]);
                            sxv[i + 1] = fmaf(kWrapMult[j], x1, sxv[i + 1]);
                        }
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float gg = gv[i];
                dwacc[i] = fmaf(hsi, gg * xav[i], dwacc[i]);
                drv[i] = fmaf(st, sxv[i], fmaf(kr, xav[i], fmaf(fmaf(brh, wv[i], a_r), gg, pr[i])));
                dbv[i] = fmaf(st, bv[i], fmaf(kb2, xav[i], fmaf(fmaf(bbh, wv[i], a_b), gg, pb[i])));
            }
            vlds_put4<TX>(out_lds[0] + boff, drv);
            vlds_put4<TX>(out_lds[1] + boff, dbv);
        }
    };
    auto store = [&](uint32_t rel) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            const int row = lrow + p * RPP;
            const uint32_t off = xo + (rel + p * RPP) * xrow;
            const uint2* pr = reinterpret_cast<const uint2*>(&out_lds[0][row * PITCH + lvec * 16]);
            const uint2* pb = reinterpret_cast<const uint2*>(&out_lds[1][row * PITCH + lvec * 16]);
            const uint2 r0 = pr[0], r1 = pr[1], b0 = pb[0], b1 = pb[1];
            buf_st16<true>(rs_dr, off, 0u, make_uint4(r0.x, r0.y, r1.x, r1.y));
            buf_st16<true>(rs_db, off, 0u, make_uint4(b0.x, b0.y, b1.x, b1.y));
        }
    };
    // stage r is in LDS, fc holds stage r + TB, fp is free
    auto step = [&](uint32_t r, Fetched& fc, Fetched& fp) __attribute__((always_inline)) {
        fetch(fp, r + DEPTH * TB);
        compute();
        __syncthreads();
        store(r);
        commit(fc);
        __syncthreads();
    };
    const uint32_t nr = (uint32_t)nrows;
    fetch(f0, 0u);
    commit(f0);
    fetch(f1, TB);
    if constexpr (DEPTH == 3) fetch(f2, 2 * TB);
    __syncthreads();
    // whole rounds of DEPTH stages: those past the last row read zeros, add
    // zeros and store nothing
    for (uint32_t r0 = 0; r0 < nr; r0 += DEPTH * TB) {
        step(r0, f1, f0);
        if constexpr (DEPTH == 3) {
            step(r0 + TB, f2, f1);
            step(r0 + 2 * TB, f0, f2);
        } else {
            step(r0 + TB, f0, f1);
        }
    }
    if (!wave_on) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) dwacc[i] = group_sum<16>(dwacc[i]);
    if (lr == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t c = cb0 + wc0 + 4 * lg + i;
            if (c < C) dw_part[(int64_t)blockIdx.y * C + c] = dwacc[i];
        }
    }
    // dphi_part[tile][stream][row][C]: row 16 m + 4 lg + i, channel wc0 + lr
    const int64_t c = cb0 + wc0 + lr;
    if (c >= C) return;
    float* out = dphi_part + (int64_t)blockIdx.y * NST * rows * C + c;
#pragma unroll
    for (int j = 0; j < NST; ++j) {
#pragma unroll
        for (int m = 0; m < MI; ++m) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int o = 16 * m + 4 * lg + i;
                if (o < rows) out[((int64_t)j * rows + o) * C] = acc[j][m][i];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// The wrapper's parameter gradients from the partials of its backward, one
// launch (WrapSums in mhc_internal.h).  Workgroups, in order:
//   dPhi  256 lanes = `phases` tile phases x columns of one (stream, row):
//         grad_phi[o][j][c] = the tiles' sum; stream 0's lanes also write the
//         streams that are its multiples (or zeros)
//   dw    the same over dw_part, in the weight's dtype
//   db, dalpha   one workgroup per column of cpart that does not vanish
//   zeros the H_res rows of dPhi, db and dalpha: s - s with s the sum of the
//         alpha gradients, so zeros that are NaN where those are not finite
// Every sum has a fixed order.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void wrap_sums_kernel(WrapSums a) {
    __shared__ float red[256];
    int bid = (int)blockIdx.x;
    auto col_sum = [&](const float* p, int64_t stride, int rows, int phases, bool on) __attribute__((always_inline)) {
        const int cpb = 256 / phases;
        const int cl = threadIdx.x % cpb, ph = threadIdx.x / cpb;
        float s = 0.f;
        if (on) {
            int r = ph;
            for (; r + 7 * phases < rows; r += 8 * phases) {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = p[(int64_t)(r + u * phases) * stride];
#pragma unroll
                for (int u = 0; u < 8; ++u) s += v[u];
            }
            for (; r < rows; r += phases) s += p[(int64_t)r * stride];
        }
        if (phases == 1) return s;
        red[threadIdx.x] = s;
        __syncthreads();
        float t = 0.f;
        if (ph == 0) {
            for (int k = 0; k < phases; ++k) t += red[k * cpb + cl];
        }
        return t;
    };
    // sum over rows of one column of cpart, the same in every lane
    auto cpart_sum = [&](int col) __attribute__((always_inline)) {
        float s = 0.f;
        for (int r = threadIdx.x; r < a.crows; r += 256) s += a.cpart[(int64_t)r * (a.np + 3) + col];
        float v[1] = {s};
        block_sum<1>(v, red);
        return v[0];
    };
    const int cpb = 256 / a.phases;
    const int cl = threadIdx.x % cpb;
    const bool first = threadIdx.x / cpb == 0;
    const int cblk = (a.C + cpb - 1) / cpb;
    const int phi_blocks = cblk * a.rows * a.nst;
    if (bid < phi_blocks) {
        const int c = (bid % cblk) * cpb + cl;
        const int o = (bid / cblk) % a.rows;
        const int j = bid / cblk / a.rows;
        const bool on = c < a.C;
        const float t = col_sum(a.phi_part + (int64_t)j * a.stream_stride + (int64_t)o * a.row_stride + (on ? c : 0),
                                a.tile_stride, a.tiles, a.phases, on);
        if (!on || !first) return;
        float* out = a.grad_phi + (int64_t)o * a.n * a.C + c;
        out[(int64_t)j * a.C] = t;
        if (j == 0) {
            double md = 1.0;
            for (int q = 2; q < a.n; ++q) {
                md *= 0.1;
                if (q >= a.nst) out[(int64_t)q * a.C] = a.decay ? (float)md * t : 0.f * t;
            }
        }
        return;
    }
    bid -= phi_blocks;
    if (bid < cblk) {
        const int c = bid * cpb + cl;
        const bool on = c < a.C;
        const float t = col_sum(a.dw_part + (on ? c : 0), a.C, a.dw_rows, a.phases, on);
        if (!on || !first) return;
        if (a.w_bf16) static_cast<bf16_t*>(a.grad_w)[c] = f32_to_bf16(t);
        else static_cast<float*>(a.grad_w)[c] = t;
        return;
    }
    bid -= cblk;
    if (a.crows == 0) return;
    if (bid < a.rows + 2) {
        const int col = bid < a.rows ? bid : a.np + (bid - a.rows);
        const float t = cpart_sum(col);
        if (threadIdx.x == 0) {
            if (bid < a.rows) a.grad_b[col] = t;
            else a.grad_alpha[bid - a.rows] = t;
        }
        return;
    }
    bid -= a.rows + 2;
    const float s0 = cpart_sum(a.np), s1 = cpart_sum(a.np + 1);
    const float z = (s0 + s1) - (s0 + s1);
    const int64_t K = (int64_t)a.n * a.C;
    float* zp = a.grad_phi + (int64_t)a.rows * K;
    const int64_t zn = (int64_t)(a.np - a.rows) * K;  // a multiple of 4, as C is
    const int64_t zi = (int64_t)bid * 256 + threadIdx.x;
    const int64_t zs = (int64_t)((int)gridDim.x - ((int)blockIdx.x - bid)) * 256;
    if ((reinterpret_cast<uintptr_t>(zp) & 15) == 0) {
        for (int64_t i = zi; i < zn / 4; i += zs) reinterpret_cast<float4*>(zp)[i] = make_float4(z, z, z, z);
    } else {
        for (int64_t i = zi; i < zn; i += zs) zp[i] = z;
    }
    if (bid == 0) {
        for (int i = threadIdx.x; i < a.np - a.rows; i += 256) a.grad_b[a.rows + i] = z;
        if (threadIdx.x == 0) a.grad_alpha[2] = z;
    }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
// bf16 'decay' past n = 8 would need a product per stream beside 2n > 16
// rows, and rows of more than 1.86M channels a tile of less than one round: those
// shapes keep the kernels of wrapper_gen.hip.
bool wbwd_shape_ok(int dt, int n, bool decay, int64_t C) {
    return n >= 2 && n <= kWgMaxN && C >= 8 && C % 8 == 0 && C <= (int64_t(1) << 21) &&
           wbwd_max_tile(C, dp_stride(2 * n + n * n)) >= kWbwdRound && (n <= 8 || dt != kBF16 || !decay);
}

int wbwd_streams(int dt, int n, bool decay) { return dt == kBF16 && decay ? n : 2; }

int wbwd_tiles(int n, int64_t B, int64_t C) {
    return (int)wbwd_split(B, C, dp_stride(2 * n + n * n), device_cu_count());
}

size_t wbwd_fold_bytes(int n, int64_t C) { return n > 8 ? (size_t)4 * n * C * sizeof(float) : 0; }

hipError_t launch_wbwd(int dt, int n, bool decay, const float* g, const void* res, const void* br, const float* w,
                       const float* ep, const float* dP, int dp_stride, const float* s_tok, const float* phi_pre,
                       const float* phi_post, float* fold, void* dres, void* dbr, float* dw_part, float* dphi_part,
                       int tiles, int64_t B, int64_t C, hipStream_t s) {
    if (B == 0) return hipSuccess;
    if (!wbwd_shape_ok(dt, n, decay, C) || tiles < 1 || (n > 8 && !fold)) return hipErrorInvalidValue;
    const int64_t tile = wbwd_tile(B, tiles);
    if (tile > wbwd_max_tile(C, dp_stride)) return hipErrorInvalidValue;
    const int Ci = (int)C;
    if (n > 8) {
        int64_t blocks = ((int64_t)2 * n * C + 255) / 256;
        if (blocks > 4096) blocks = 4096;
        MHC_LAUNCH_GGL(wbwd_fold_phi_kernel, dim3((unsigned)blocks), dim3(256), 0, s, phi_pre, phi_post, n, Ci,
                       decay ? 1 : 0, fold);
    } else {
        fold = nullptr;
    }
    // sum_j w_j^2 over the streams of r that the kernel does not form itself
    const bool xs = dt == kBF16 && decay && n > 2;
    double sq = 1.0, m = 1.0;
    if (decay) {
        for (int j = 2; j < n; ++j) {
            m *= 0.1;
            if (!xs || j >= 4) sq += (double)(float)m * (double)(float)m;
        }
    }
    const float wsq = (float)sq;
    const int dec = decay ? 1 : 0;
    const dim3 grid((unsigned)((C + kVbCols - 1) / kVbCols), (unsigned)tiles);
    const int tok = timing_begin("wrap_proj_bwd", s);
#define MHC_VB(TX_, NST_, MI_)                                                                                       \
    MHC_LAUNCH_GGL((wbwd_kernel<TX_, NST_, MI_>), grid, dim3(kVbThreads), 0, s, g, (const TX_*)res, (const TX_*)br, w, \
                   ep, dP, dp_stride, s_tok, phi_pre, phi_post, (const float*)fold, n, dec, wsq, (TX_*)dres, (TX_*)dbr, \
                   dw_part, dphi_part, B, Ci, tile)
#define MHC_VB_MI(TX_)                 \
    if (n <= 8) {                      \
        MHC_VB(TX_, 2, 1);             \
    } else if (n <= 16) {              \
        MHC_VB(TX_, 2, 2);             \
    } else {                           \
        MHC_VB(TX_, 2, 4);             \
    }
    if (dt != kBF16) {
        MHC_VB_MI(float)
    } else if (!xs) {
        MHC_VB_MI(bf16_t)
    } else {
        switch (n) {
            case 3: MHC_VB(bf16_t, 3, 1); break;
            case 4: MHC_VB(bf16_t, 4, 1); break;
            case 5: MHC_VB(bf16_t, 5, 1); break;
            case 6: MHC_VB(bf16_t, 6, 1); break;
            case 7: MHC_VB(bf16_t, 7, 1); break;
            default: MHC_VB(bf16_t, 8, 1); break;
        }
    }
#undef MHC_VB_MI
#undef MHC_VB
    timing_end(tok, s);
    return hipGetLastError();
}

hipError_t launch_wrap_sums(WrapSums a, hipStream_t s) {
    if (a.tiles < 1 || a.dw_rows < 1 || a.C < 4 || a.C % 4 != 0 || a.rows < 1 || a.nst < 2 || a.nst > a.n ||
        (a.crows > 0 && a.rows >= a.np))
        return hipErrorInvalidValue;
    const int most = a.tiles > a.dw_rows ? a.tiles : a.dw_rows;
    a.phases = most <= 8 ? 1 : (most <= 64 ? 2 : 4);
    const int cpb = 256 / a.phases;
    const int64_t cblk = (a.C + cpb - 1) / cpb;
    int64_t blocks = cblk * a.rows * a.nst + cblk;
    if (a.crows > 0) {
        // zero rows: 64 KB a workgroup, at most two per CU (each first sums the
        // alpha columns)
        int64_t zb = (int64_t)(a.np - a.rows) * a.n * a.C / 16384;
        const int64_t cap = 2 * (int64_t)device_cu_count();
        if (zb > cap) zb = cap;
        blocks += a.rows + 2 + (zb < 1 ? 1 : zb);
    }
    if (blocks > 0x7fffffff) return hipErrorInvalidValue;
    MHC_LAUNCH_GGL(wrap_sums_kernel, dim3((unsigned)blocks), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace mhc
