// Forward projection of the MHCResidualWrapper's streams (layer.py:299-310,
// ops.py:272-315), P = X Phi^T and sum X^2 per token with
// X = (r, b, w_2 r, w_3 r, ..) and w_j = 0.1^(j-1) ('decay') or 0 ('zero'),
// without a product per stream: since the streams past the second are
// multiples of r up to their rounding to the storage type,
//   P = r . Phi_r + b . Phi_1 + sum_j d_j . Phi_j,
//   Phi_r = Phi_0 + sum_{j >= 2} w_j Phi_j (fp32),   d_j = X_j - w_j r.
// With fp32 storage d_j is below the fp32 rounding of the r term and is
// dropped with it; 'zero' has no further streams.  With bf16 storage |d_j| <=
// 2^-9 w_j |r|, so a product of the bf16 parts of d_j and Phi_j, off by 2^-9 of
// it, is below the r term's fp32 rounding (2^-24) from stream 3 on (2^-18 w_j,
// w_3 = 0.01); stream 2 takes d_h Phi_h + d_h Phi_m + d_m Phi_h (2^-17 of it).
// Past w_j = 1e-4 (stream 5) d_j itself is below (2^-9 1e-5) and is dropped.
// n = 8: 12 plane products instead of 24 for each element of r, and two streams'
// worth of 'k' instead of eight at any n.
//
// The products run on bf16 MFMA 16x16x32, D[output][token]: A = Phi planes, B
// = the token rows.  Phi_r and Phi_1 are split hi / mid / lo (exact to fp32);
// fp32 rows are split hi / mid / lo in registers and their products keep the
// six terms of 2^-16 and above.  The products below hi . hi have an accumulator
// of their own where the registers allow it (wp_two_acc).
//
// A wave owns 16 TW tokens and all RT output tiles of its row block: each Phi
// fragment (1 KB of LDS) feeds TW MFMAs, and a token's d_j fragments are built
// once.  The rows go from memory straight to the fragment registers: with bf16 a
// lane's k order is free as long as Phi is packed alike, so lane group g of a
// 64-channel stage takes channels 16 g .. 16 g + 15 of its token (two 16-byte
// loads, four groups a whole 128-byte line).  Phi planes go through LDS, one
// 32-channel step ahead of the MFMAs, packed so that a step of a row block is one
// contiguous run.
// Measured (n = 8, 65,536 tokens x 7168 bf16; the rows are 1.9 GB): 3532 us for
// the eight rebuilt streams through the layer's streaming projection, 1392 us
// folded with four waves of unrolled planes (376 registers, one wave per SIMD:
// the residual arithmetic and the MFMAs took turns), 980 us with eight waves; with
// the residual streams formed in each product of stream 2 1260.  It follows the vector
// work of the residual streams as well as the MFMAs.
// Error of P against float64 (rms, relative; 3 draws each): n = 3..32, 32 to
// 2100 tokens, 64 to 7168 channels 0.65e-7 to 3.4e-7, 0.25 to 0.98 of that of the
// unfolded form on the same inputs; with one accumulator and one plane for stream
// 2, 865 us here, it was up to 2.5 times the unfolded form's (n = 3, 700 x 512:
// 2.9e-7 for 1.2e-7, 1.0e-7 now).
#include "mhc_device.h"
#include "mhc_internal.h"
#include "wrapper_plan.h"

namespace mhc {

namespace {

typedef __bf16 wbf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 wbf16x2_t __attribute__((ext_vector_type(2)));
typedef float wf32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int wu32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ wf32x4_t wmfma(wu32x4_t a, wu32x4_t b, wf32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(wbf16x8_t, a), __builtin_bit_cast(wbf16x8_t, b),
                                                   c, 0, 0, 0);
}

// c + a.x b.x + a.y b.y of packed bf16 pairs (products exact, fp32 sums)
__device__ __forceinline__ float wdot2(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(wbf16x2_t, a), __builtin_bit_cast(wbf16x2_t, b), c, false);
}

__device__ __forceinline__ float wlo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float whi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// 0.1^(j-1) as Python's product gives it in fp32
constexpr double wp_pow01(int e) { return e <= 0 ? 1.0 : 0.1 * wp_pow01(e - 1); }
constexpr float kWpMult[7] = {1.f, 0.f, (float)wp_pow01(1), (float)wp_pow01(2), (float)wp_pow01(3),
                              (float)wp_pow01(4), (float)wp_pow01(5)};
// kWpMult[j] of a wave-uniform j in 2..6, as scalar selects
__device__ __forceinline__ float wp_mult(int j) {
    float m = kWpMult[2];
    m = j == 3 ? kWpMult[3] : m;
    m = j == 4 ? kWpMult[4] : m;
    m = j == 5 ? kWpMult[5] : m;
    return j == 6 ? kWpMult[6] : m;
}

constexpr int kWpMaxRes = 4;  // residual streams 2 .. 5 (bf16 'decay')

// Planes of Phi of a step: r and b hi / mid / lo, then -Phi_j of each residual
// stream (the kernel forms w r - X), the first of them hi / mid.
constexpr int wp_planes(int nres) { return 6 + nres + (nres > 0 ? 1 : 0); }

// Products of two hi parts and the smaller ones in accumulators of their own:
// then a step rounds the large sum twice and not 6 to 13 times.  Where the
// registers allow it (bf16 rows at 64 tokens a wave: 256 of them, up to three
// row tiles; past that the long chains of the same tokens are no shorter in any
// other form).
constexpr bool wp_two_acc(bool bf16, int rt, int tw) { return !bf16 || rt * tw <= 12; }

}  // namespace

// ---------------------------------------------------------------------------
// Phi -> planes in A-fragment order.  Step hs covers 32 of the channels: bf16
// rows take them in the order described above (lane group g of half h of the
// 64-channel stage s: channels 64 s + 16 g + 8 h ..), fp32 rows in order
// (32 hs + 8 g ..).
//   out[(((rb * steps + hs) * NPL + p) * RT + rt) * 64 + lane]   (16 bytes)
// = plane p of row o = (rb RT + rt) 16 + lane % 16, zero past np and past C.
// One lane per fragment position, all planes; the same launch converts the
// RMSNorm weight to fp32.
// ---------------------------------------------------------------------------
template <bool BF16>
__global__ __launch_bounds__(256) void wfold_pack_kernel(const float* __restrict__ pre, const float* __restrict__ post,
                                                         const float* __restrict__ resm, int n, int np, int C,
                                                         int decay, int nres, int RT, int row_blocks, int steps,
                                                         uint4* __restrict__ out, const void* __restrict__ weight,
                                                         int w_dtype, float* __restrict__ w32) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (int64_t c = gid; c < C; c += stride)
        w32[c] = w_dtype == kBF16 ? bf16_to_f32(static_cast<const bf16_t*>(weight)[c])
                                  : static_cast<const float*>(weight)[c];
    const int npl = wp_planes(nres);
    const int64_t K = (int64_t)n * C;
    const int64_t total = (int64_t)row_blocks * steps * RT * 64;
    for (int64_t i = gid; i < total; i += stride) {
        const int lane = (int)(i & 63);
        const int64_t q = i >> 6;
        const int rt = (int)(q % RT);
        const int hs = (int)((q / RT) % steps);
        const int rb = (int)(q / RT / steps);
        const int g = lane >> 4;
        const int o = (rb * RT + rt) * 16 + (lane & 15);
        const int c0 = BF16 ? 64 * (hs >> 1) + 16 * g + 8 * (hs & 1) : 32 * hs + 8 * g;
        const bool ok = o < np && c0 < C;  // C % 8 == 0: the 8 channels are in or out
        const float* row = ok ? phi_row(pre, post, resm, n, o, K) + c0 : pre;
        uint4* dst = out + (((int64_t)(rb * steps + hs) * npl) * RT + rt) * 64 + lane;
        auto put = [&](int p, const float (&v)[8]) __attribute__((always_inline)) {
            dst[(int64_t)p * RT * 64] = make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]),
                                                   pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
        };
        auto put3 = [&](int p, float (&v)[8]) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                put(p + k, v);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] -= bf16_to_f32(f32_to_bf16(v[e]));
            }
        };
        float vr[8], v[8];
        auto ld = [&](int j, float (&d)[8]) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < 8; ++e) d[e] = 0.f;
            if (ok) load_run<float, 8>(row + (int64_t)j * C, d);
        };
        ld(0, vr);
        double md = 1.0;
        for (int j = 2; j < n; ++j) {
            md *= 0.1;
            const float m = decay ? (float)md : 0.f;  // (0 Phi_j: NaN where Phi_j is not finite, as X_j Phi_j is)
            ld(j, v);
#pragma unroll
            for (int e = 0; e < 8; ++e) vr[e] = fmaf(m, v[e], vr[e]);
            if (j - 2 < nres) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = -v[e];
                put(j == 2 ? 6 : 5 + j, v);
                if (j == 2) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] -= bf16_to_f32(f32_to_bf16(v[e]));
                    put(7, v);
                }
            }
        }
        put3(0, vr);
        ld(1, v);
        put3(3, v);
    }
}

// ---------------------------------------------------------------------------
// P partials [tile of 32 rows][split][B][32] and sum X^2 partials [split][B]
// (the coefficient kernels' layout).  Workgroup = wp_waves(TW) waves x 16 TW tokens;
// grid x = token blocks x the rbs row blocks of RT 16-row tiles (fastest, so
// that the row blocks of a token block run together and share its rows in
// L2); y = ks channel splits of `schunk` steps (even for bf16).
// ---------------------------------------------------------------------------
template <typename TX, int RT, int NRES, int TW>
__global__ __launch_bounds__(64 * wp_waves(sizeof(TX), TW)) void wfold_proj_kernel(const TX* __restrict__ res, const TX* __restrict__ br,
                                                                const uint4* __restrict__ phi,
                                                                float* __restrict__ p_part,
                                                                float* __restrict__ ss_part, int64_t B, int C, int np,
                                                                int steps, int schunk, int ks, int rbs, float wsq) {
    constexpr bool BF = sizeof(TX) == 2;
    constexpr int kWpWaves = wp_waves(sizeof(TX), TW);
    constexpr int NPL = wp_planes(NRES);
    constexpr int CH = NPL * RT;                        // 1 KB fragments of a step
    constexpr int CPW = (CH + kWpWaves - 1) / kWpWaves;  // staged by a wave
    static_assert(BF || NRES == 0, "residual streams are bf16 rows'");
    __shared__ __align__(16) wu32x4_t phl[2][CH * 64];
    const int lane = threadIdx.x & 63;
    const int wave = (int)wave_uniform(threadIdx.x >> 6);
    const int lr = lane & 15;
    const int g = lane >> 4;
    const int rb = (int)(blockIdx.x % rbs);
    const int q = blockIdx.y;
    const int h0 = q * schunk;
    const int h1 = h0 + schunk < steps ? h0 + schunk : steps;
    const int64_t t0 = ((int64_t)(blockIdx.x / rbs) * kWpWaves + wave) * (16 * TW);
    const int64_t nrows = t0 < B ? (B - t0 < 16 * TW ? B - t0 : 16 * TW) : 0;
    const int64_t tb = nrows > 0 ? t0 : 0;
    const uint32_t rowb = (uint32_t)C * (uint32_t)sizeof(TX);
    const buf_rsrc_t rs_r = make_buf_rsrc(res + tb * C, (uint32_t)nrows * rowb);
    const buf_rsrc_t rs_b = make_buf_rsrc(br + tb * C, (uint32_t)nrows * rowb);
    const wu32x4_t* pw = reinterpret_cast<const wu32x4_t*>(phi) + ((int64_t)rb * steps) * CH * 64 + lane;

    constexpr bool TWO = wp_two_acc(BF, RT, TW);
    wf32x4_t acc[RT][TW], accs[TWO ? RT : 1][TWO ? TW : 1];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
        for (int tt = 0; tt < TW; ++tt) {
            acc[rt][tt] = wf32x4_t{0.f, 0.f, 0.f, 0.f};
            if constexpr (TWO) accs[rt][tt] = acc[rt][tt];
        }
    }
    // the accumulator of the products below hi . hi
    auto small = [&](int rt, int tt) __attribute__((always_inline)) -> wf32x4_t& {
        if constexpr (TWO) {
            return accs[rt][tt];
        } else {
            return acc[rt][tt];
        }
    };
    // (-1, 0) and (0, -1), held in registers: as a literal operand of the dot
    // product the first becomes the inline constant -1.0, which the hardware
    // reads as its fp32 bits, (0, -1)
    uint32_t neg_lo = 0x0000bf80u, neg_hi = 0xbf800000u;
    asm volatile("" : "+v"(neg_lo), "+v"(neg_hi));
    float ss[TW], sb[TW];
#pragma unroll
    for (int tt = 0; tt < TW; ++tt) ss[tt] = sb[tt] = 0.f;

    // the wave's rows of one step: bf16 one 16-byte piece per token tile and
    // array, fp32 two.  Pieces past C (and tokens past B) read zeros.
    constexpr int PC = BF ? 1 : 2;
    struct Rows {
        uint4 r[TW][PC], b[TW][PC];
    };
    auto fetch = [&](Rows& f, int hs) __attribute__((always_inline)) {
        const int c = BF ? 64 * (hs >> 1) + 16 * g + 8 * (hs & 1) : 32 * hs + 8 * g;
        const bool ok = c < C && hs < h1;
        const uint32_t o0 = (uint32_t)lr * rowb + (uint32_t)c * (uint32_t)sizeof(TX);
#pragma unroll
        for (int tt = 0; tt < TW; ++tt) {
#pragma unroll
            for (int p = 0; p < PC; ++p) {
                const uint32_t o = ok ? o0 + (uint32_t)(16 * tt) * rowb + 16u * p : kBufOff;
                f.r[tt][p] = buf_ld16<false, true>(rs_r, o, 0u);
                f.b[tt][p] = buf_ld16<false, true>(rs_b, o, 0u);
            }
        }
    };
    wu32x4_t st[CPW];
    auto fetch_phi = [&](int hs) __attribute__((always_inline)) {
        const int h = hs < h1 ? hs : h0;  // past the split's last step: any step's planes (h0 < steps)
#pragma unroll
        for (int k = 0; k < CPW; ++k) {
            const int c = wave + kWpWaves * k;
            st[k] = pw[((int64_t)h * CH + (c < CH ? c : 0)) * 64];
        }
    };
    auto commit_phi = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < CPW; ++k) {
            const int c = wave + kWpWaves * k;
            if (c < CH) phl[buf][c * 64 + lane] = st[k];
        }
    };
    auto frag = [&](int buf, int p, int rt) __attribute__((always_inline)) -> wu32x4_t {
        return phl[buf][(p * RT + rt) * 64 + lane];
    };
    auto step = [&](const Rows& f, int buf) __attribute__((always_inline)) {
        if constexpr (BF) {
            wu32x4_t xr[TW], xb[TW];
#pragma unroll
            for (int tt = 0; tt < TW; ++tt) {
                const uint4 r = f.r[tt][0], b = f.b[tt][0];
                xr[tt] = wu32x4_t{r.x, r.y, r.z, r.w};
                xb[tt] = wu32x4_t{b.x, b.y, b.z, b.w};
            }
            // rolled loops: one plane's products at a time keep the wave within
            // 256 registers (two waves per SIMD)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const wu32x4_t a = frag(buf, 0, rt);
#pragma unroll
                for (int tt = 0; tt < TW; ++tt) acc[rt][tt] = wmfma(a, xr[tt], acc[rt][tt]);
            }
#pragma unroll 1
            for (int p = 1; p < 3; ++p) {
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    const wu32x4_t a = frag(buf, p, rt);
#pragma unroll
                    for (int tt = 0; tt < TW; ++tt) small(rt, tt) = wmfma(a, xr[tt], small(rt, tt));
                }
            }
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const wu32x4_t a = frag(buf, 3, rt);
#pragma unroll
                for (int tt = 0; tt < TW; ++tt) acc[rt][tt] = wmfma(a, xb[tt], acc[rt][tt]);
            }
#pragma unroll 1
            for (int p = 4; p < 6; ++p) {
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    const wu32x4_t a = frag(buf, p, rt);
#pragma unroll
                    for (int tt = 0; tt < TW; ++tt) small(rt, tt) = wmfma(a, xb[tt], small(rt, tt));
                }
            }
#pragma unroll
            for (int tt = 0; tt < TW; ++tt) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    ss[tt] = wdot2(xr[tt][e], xr[tt][e], ss[tt]);
                    ss[tt] = wdot2(xb[tt][e], xb[tt][e], ss[tt]);
                }
            }
            // w r - X of a stream, exact: -d_j (the packed planes are -Phi_j), and
            // its bf16 part; X^2 into sq
            auto resid = [&](uint32_t xw, float m, bool add, float& sq, float& d0, float& d1)
                __attribute__((always_inline)) {
                const float p0 = wlo(xw) * m, p1 = whi(xw) * m;
                const uint32_t x = pack_bf16x2(p0, p1);  // the stored stream
                const uint32_t xs = add ? x : 0u;
                sq = wdot2(xs, xs, sq);
                d0 = wdot2(x, neg_lo, p0);
                d1 = wdot2(x, neg_hi, p1);
                return pack_bf16x2(d0, d1);
            };
            // stream 2, whose rounding is the largest: -d_2 and Phi_2 hi + mid
            constexpr bool ONE = NRES > 0 && RT * TW >= 24;
            if constexpr (NRES > 0 && !ONE) {
                wu32x4_t dh[TW], dm[TW];
#pragma unroll
                for (int tt = 0; tt < TW; ++tt) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float d0, d1;
                        dh[tt][e] = resid(xr[tt][e], kWpMult[2], true, ss[tt], d0, d1);
                        dm[tt][e] = pack_bf16x2(wdot2(dh[tt][e], neg_lo, d0), wdot2(dh[tt][e], neg_hi, d1));
                    }
                }
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    const wu32x4_t a = frag(buf, 6, rt), am = frag(buf, 7, rt);
#pragma unroll
                    for (int tt = 0; tt < TW; ++tt) small(rt, tt) = wmfma(a, dh[tt], small(rt, tt));
#pragma unroll
                    for (int tt = 0; tt < TW; ++tt) small(rt, tt) = wmfma(am, dh[tt], small(rt, tt));
#pragma unroll
                    for (int tt = 0; tt < TW; ++tt) small(rt, tt) = wmfma(a, dm[tt], small(rt, tt));
                }
            }
            // the others, one plane each; with six row tiles, where both parts of
            // d_2 do not fit, its three products first (t = 0, 1, 2)
#pragma unroll 1
            for (int t = ONE ? 0 : 3; t < NRES + 2; ++t) {
                const float m = t < 3 ? kWpMult[2] : wp_mult(t);
                const bool low = ONE && t == 2, again = ONE && (t == 1 || t == 2);
                wu32x4_t d[TW];
#pragma unroll
                for (int tt = 0; tt < TW; ++tt) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float d0, d1;
                        const uint32_t h = resid(xr[tt][e], m, !again, ss[tt], d0, d1);
                        if constexpr (ONE) {
                            d0 -= low ? wlo(h) : 0.f;
                            d1 -= low ? whi(h) : 0.f;
                            d[tt][e] = pack_bf16x2(d0, d1);
                        } else {
                            d[tt][e] = h;
                        }
                    }
                }
                const int p = low ? 6 : (t < 3 ? 6 + t : 5 + t);
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    const wu32x4_t a = frag(buf, p, rt);
#pragma unroll
                    for (int tt = 0; tt < TW; ++tt) small(rt, tt) = wmfma(a, d[tt], small(rt, tt));
                }
            }
        } else {
            // split each operand hi / mid / lo; products of weight 2^-16 and above
            wu32x4_t x3[3][TW];
#pragma unroll
            for (int a2 = 0; a2 < 2; ++a2) {
#pragma unroll
                for (int tt = 0; tt < TW; ++tt) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint4 w = a2 == 0 ? f.r[tt][e / 2] : f.b[tt][e / 2];
                        float v0 = __uint_as_float(e % 2 == 0 ? w.x : w.z), v1 = __uint_as_float(e % 2 == 0 ? w.y : w.w);
                        float& s = a2 == 0 ? ss[tt] : sb[tt];
                        s = fmaf(v0, v0, s);
                        s = fmaf(v1, v1, s);
                        const uint32_t h = pack_bf16x2(v0, v1);
                        v0 -= wlo(h);
                        v1 -= whi(h);
                        const uint32_t m = pack_bf16x2(v0, v1);
                        v0 -= wlo(m);
                        v1 -= whi(m);
                        x3[0][tt][e] = h;
                        x3[1][tt][e] = m;
                        x3[2][tt][e] = pack_bf16x2(v0, v1);
                    }
                }
#pragma unroll
                for (int p = 0; p < 3; ++p) {
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt) {
                        const wu32x4_t a = frag(buf, 3 * a2 + p, rt);
#pragma unroll
                        for (int k = 0; k < 3 - p; ++k) {
#pragma unroll
                            for (int tt = 0; tt < TW; ++tt) {
                                wf32x4_t& c = p + k == 0 ? acc[rt][tt] : small(rt, tt);
                                c = wmfma(a, x3[k][tt], c);
                            }
                        }
                    }
                }
            }
        }
    };

    // Rows of steps hs and hs + 1 alternate between two register sets: a set
    // is refilled as soon as its step's products are issued, one step before
    // its next use.  Phi of step hs + 1 is fetched while step hs computes and
    // committed to the other LDS buffer; one barrier per step.
    Rows f0, f1;
    fetch(f0, h0);
    fetch(f1, h0 + 1);
    fetch_phi(h0);
    commit_phi(0);
    __syncthreads();
    for (int hs = h0; hs < h1; hs += 2) {
        fetch_phi(hs + 1);
        step(f0, 0);
        fetch(f0, hs + 2);
        commit_phi(1);
        __syncthreads();
        fetch_phi(hs + 2);
        if (hs + 1 < h1) step(f1, 1);  // the same for the whole grid row
        fetch(f1, hs + 3);
        commit_phi(0);
        __syncthreads();
    }

    if constexpr (TWO) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
            for (int tt = 0; tt < TW; ++tt) acc[rt][tt] += accs[rt][tt];
        }
    }
    // lane: token lr of tile tt, outputs 4 g .. 4 g + 3 of row tile rt
    const int tiles = (np + kProjTile - 1) / kProjTile;
#pragma unroll
    for (int tt = 0; tt < TW; ++tt) {
        const int64_t tok = t0 + 16 * tt + lr;
        if (tok < B) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const int o = (rb * RT + rt) * 16 + 4 * g;
                if ((o >> 5) < tiles)
                    *reinterpret_cast<float4*>(p_part + (((int64_t)(o >> 5) * ks + q) * B + tok) * kProjTile + (o & 31)) =
                        make_float4(acc[rt][tt][0], acc[rt][tt][1], acc[rt][tt][2], acc[rt][tt][3]);
            }
        }
        float s = BF ? ss[tt] : fmaf(ss[tt], wsq, sb[tt]);
        s = xor32_add(xor16_add(s));
        if (rb == 0 && g == 0 && tok < B) ss_part[(int64_t)q * B + tok] = s;
    }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
static int wfold_nres(int dt, int n, bool decay) {
    if (dt != kBF16 || !decay) return 0;
    return n - 2 < kWpMaxRes ? n - 2 : kWpMaxRes;
}

int wfold_ksplit(int dt, int64_t B, int64_t C, int np) {
    return wfold_split(dt == kBF16, B, C, np, device_cu_count()).ks;
}

size_t wfold_pack_bytes(int dt, int n, int64_t C, int np) {
    return (size_t)wfold_row_blocks(np) * wfold_steps(dt == kBF16, C) * wp_planes(wfold_nres(dt, n, true)) *
           wfold_rt(np) * 1024;
}

bool wfold_ok(int n, int64_t C) { return n >= 2 && n <= kWgMaxN && C >= 8 && C % 8 == 0 && C <= (int64_t(1) << 21); }

// Rows at an address that is not 16-byte aligned, moved to one that is.
template <typename T>
__global__ __launch_bounds__(256) void wfold_copy_kernel(const T* __restrict__ a, T* __restrict__ ao,
                                                         const T* __restrict__ b, T* __restrict__ bo, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        ao[i] = a[i];
        bo[i] = b[i];
    }
}

hipError_t launch_wfold_copy(int dt, const void* res, void* res_out, const void* br, void* br_out, int64_t elems,
                             hipStream_t s) {
    if (elems == 0) return hipSuccess;
    int64_t blocks = (elems + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    if (dt == kBF16) {
        MHC_LAUNCH_GGL(wfold_copy_kernel<bf16_t>, dim3((unsigned)blocks), dim3(256), 0, s, (const bf16_t*)res,
                       (bf16_t*)res_out, (const bf16_t*)br, (bf16_t*)br_out, elems);
    } else {
        MHC_LAUNCH_GGL(wfold_copy_kernel<float>, dim3((unsigned)blocks), dim3(256), 0, s, (const float*)res,
                       (float*)res_out, (const float*)br, (float*)br_out, elems);
    }
    return hipGetLastError();
}

template <typename TX, int RT, int NRES>
static void wfold_launch(int tw, dim3 grid, hipStream_t s, const void* res, const void* br, const uint4* phi,
                         float* p_part, float* ss_part, int64_t B, int C, int np, int steps, int schunk, int ks,
                         int rbs, float wsq) {
#define MHC_WF_TW(TW_)                                                                                               \
    MHC_LAUNCH_GGL((wfold_proj_kernel<TX, RT, NRES, TW_>), grid, dim3(64 * wp_waves(sizeof(TX), TW_)), 0, s, (const TX*)res, (const TX*)br, \
                   phi, p_part, ss_part, B, C, np, steps, schunk, ks, rbs, wsq)
    if (tw == 4) {
        MHC_WF_TW(4);
    } else if (tw == 2) {
        MHC_WF_TW(2);
    } else {
        MHC_WF_TW(1);
    }
#undef MHC_WF_TW
}

hipError_t launch_wfold_proj(int dt, int n, bool decay, const void* res, const void* br, const float* phi_pre,
                             const float* phi_post, const float* phi_res, const void* weight, int w_dtype, float* w32,
                             void* pack, float* p_part, float* ss_part, int64_t B, int64_t C, int ks, hipStream_t s) {
    if (B == 0) return hipSuccess;
    const int np = 2 * n + n * n;
    if (!wfold_ok(n, C) || ks < 1 || reinterpret_cast<uintptr_t>(res) % 16 != 0 ||
        reinterpret_cast<uintptr_t>(br) % 16 != 0)
        return hipErrorInvalidValue;
    const int nres = wfold_nres(dt, n, decay), rt = wfold_rt(np);
    const int rbs = wfold_row_blocks(np);
    const WfoldSplit sp = wfold_split(dt == kBF16, B, C, np, device_cu_count());
    // (the kernel's prologue reads the first step of its split)
    if (ks != sp.ks || (int64_t)(sp.ks - 1) * sp.chunk >= sp.steps) return hipErrorInvalidValue;
    const int steps = sp.steps, schunk = sp.chunk;
    const int Ci = (int)C;
    const int64_t frags = (int64_t)rbs * steps * rt * 64;
    int64_t pblocks = (frags + 255) / 256;
    if (pblocks > 8192) pblocks = 8192;
    if (dt == kBF16) {
        MHC_LAUNCH_GGL(wfold_pack_kernel<true>, dim3((unsigned)pblocks), dim3(256), 0, s, phi_pre, phi_post, phi_res, n,
                       np, Ci, decay ? 1 : 0, nres, rt, rbs, steps, (uint4*)pack, weight, w_dtype, w32);
    } else {
        MHC_LAUNCH_GGL(wfold_pack_kernel<false>, dim3((unsigned)pblocks), dim3(256), 0, s, phi_pre, phi_post, phi_res,
                       n, np, Ci, decay ? 1 : 0, nres, rt, rbs, steps, (uint4*)pack, weight, w_dtype, w32);
    }
    const int tw = wfold_tw(B);
    const int64_t per = wfold_tokens(dt == kBF16, B);
    const int64_t gx = (B + per - 1) / per * rbs;
    if (gx > 0x7fffffff || ks > 65535) return hipErrorInvalidValue;
    const dim3 grid((unsigned)gx, (unsigned)ks);
    double sq = 1.0;  // sum_j w_j^2 over r's streams (fp32 rows)
    if (decay) {
        double m = 1.0;
        for (int j = 2; j < n; ++j) {
            m *= 0.1;
            sq += (double)(float)m * (double)(float)m;
        }
    }
    const float wsq = (float)sq;
    const uint4* ph = (const uint4*)pack;
    const int tok = timing_begin("proj", s);
#define MHC_WF(TX_, RT_, NR_)                                                                                         \
    wfold_launch<TX_, RT_, NR_>(tw, grid, s, res, br, ph, p_part, ss_part, B, Ci, np, steps, schunk, ks, rbs, wsq)
#define MHC_WF_RT(TX_)                       \
    switch (rt) {                            \
        case 1: MHC_WF(TX_, 1, 0); break;    \
        case 2: MHC_WF(TX_, 2, 0); break;    \
        case 3: MHC_WF(TX_, 3, 0); break;    \
        case 4: MHC_WF(TX_, 4, 0); break;    \
        case 5: MHC_WF(TX_, 5, 0); break;    \
        default: MHC_WF(TX_, 6, 0); break;   \
    }
    if (dt != kBF16) {
        MHC_WF_RT(float)
    } else if (nres == 0) {
        MHC_WF_RT(bf16_t)
    } else if (nres == 1) {  // n = 3: 15 rows
        MHC_WF(bf16_t, 1, 1);
    } else if (nres == 2) {  // n = 4: 24 rows
        MHC_WF(bf16_t, 2, 2);
    } else if (nres == 3) {  // n = 5: 35 rows
        MHC_WF(bf16_t, 3, 3);
    } else {  // n >= 6: 48 rows and more
        switch (rt) {
            case 3: MHC_WF(bf16_t, 3, 4); break;
            case 4: MHC_WF(bf16_t, 4, 4); break;
            case 5: MHC_WF(bf16_t, 5, 4); break;
            default: MHC_WF(bf16_t, 6, 4); break;
        }
    }
#undef MHC_WF_RT
#undef MHC_WF
    timing_end(tok, s);
    return hipGetLastError();
}

}  // namespace mhc
