// xtern: the elementwise middle of the MLP block (activation, optional
// RMSNorm, requantisation), also xt_activation_mul and xt_rms_norm (gfx950).
//
// Reference behaviour: silu_inplace (src/bit1_58/quantization.rs:201-286),
// FastTensor::silu_mul_inplace / relu2_mul_inplace / rmsnorm
// (src/tensor.rs:170-265), rms_norm (src/nn/fast_attention_simd.rs:458-516).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/xtern.h"
#include "xtern_device.h"
#include "xtern_internal.h"

namespace xt {

// expf of the C library the reference links (glibc 2.28+, from ARM's
// optimized-routines): x * 32/ln2 rounded to an integer k, 2^(k/32) from a
// 32-entry table with k/32's integer part added to the exponent bits, and a
// cubic in the remainder, all in double, rounded once to float.  The two
// products with InvLn2N are fused multiply-adds, as the FMA build of the
// library compiles them.  Equal to the host expf on every one of the 2^32
// float inputs (checked exhaustively on the build host).
__constant__ uint64_t kExp2Tab[32] = {
    0x3ff0000000000000ULL, 0x3fefd9b0d3158574ULL, 0x3fefb5586cf9890fULL, 0x3fef9301d0125b51ULL,
    0x3fef72b83c7d517bULL, 0x3fef54873168b9aaULL, 0x3fef387a6e756238ULL, 0x3fef1e9df51fdee1ULL,
    0x3fef06fe0a31b715ULL, 0x3feef1a7373aa9cbULL, 0x3feedea64c123422ULL, 0x3feece086061892dULL,
    0x3feebfdad5362a27ULL, 0x3feeb42b569d4f82ULL, 0x3feeab07dd485429ULL, 0x3feea47eb03a5585ULL,
    0x3feea09e667f3bcdULL, 0x3fee9f75e8ec5f74ULL, 0x3feea11473eb0187ULL, 0x3feea589994cce13ULL,
    0x3feeace5422aa0dbULL, 0x3feeb737b0cdc5e5ULL, 0x3feec49182a3f090ULL, 0x3feed503b23e255dULL,
    0x3feee89f995ad3adULL, 0x3feeff76f2fb5e47ULL, 0x3fef199bdd85529cULL, 0x3fef3720dcef9069ULL,
    0x3fef5818dcfba487ULL, 0x3fef7c97337b9b5fULL, 0x3fefa4afa2a490daULL, 0x3fefd0765b6e4540ULL};

__device__ __forceinline__ float libc_expf(float x) {
    const uint32_t ux = __float_as_uint(x);
    const uint32_t top = (ux >> 20) & 0x7ffu;
    if (top >= 0x42bu) {  // |x| >= 88, inf, NaN
        if (ux == 0xff800000u) return 0.0f;
        if (top >= 0x7f8u) return x + x;
        if (x > 0x1.62e42ep6f) return __builtin_inff();
        if (x < -0x1.9fe368p6f) return 0.0f;
    }
    const double C0 = 0x1.c6af84b912394p-5 / 32 / 32 / 32, C1 = 0x1.ebfce50fac4f3p-3 / 32 / 32,
                 C2 = 0x1.62e42ff0c52d6p-1 / 32;
    const double inv = 0x1.71547652b82fep+0 * 32, shift = 0x1.8p+52;
    const double xd = (double)x;
    double kd = __fma_rn(inv, xd, shift);
    const uint64_t ki = (uint64_t)__double_as_longlong(kd);
    kd = __dsub_rn(kd, shift);
    const double r = __fma_rn(inv, xd, -kd);
    const uint64_t t = kExp2Tab[ki & 31] + (ki << 47);
    const double s = __longlong_as_double((long long)t);
    const double z = __fma_rn(C0, r, C1);
    const double r2 = __dmul_rn(r, r);
    double y = __fma_rn(C2, r, 1.0);
    y = __fma_rn(z, r2, y);
    return (float)__dmul_rn(y, s);
}

// quantization.rs:213 / :280: g * (1 / (1 + exp(-g))) * u.
__device__ __forceinline__ float silu_scalar(float g, float u) {
    const float sig = __fdiv_rn(1.0f, __fadd_rn(1.0f, libc_expf(-g)));
    return __fmul_rn(__fmul_rn(g, sig), u);
}
// tensor.rs:186-188: (x / (1 + exp(-x))) * u.
__device__ __forceinline__ float silu_div(float g, float u) {
    return __fmul_rn(__fdiv_rn(g, __fadd_rn(1.0f, libc_expf(-g))), u);
}
// quantization.rs:215-216, :268-270; tensor.rs:223-224: max(g, 0)^2 * u.
__device__ __forceinline__ float relu2_mul(float g, float u) {
    const float r = (g > 0.0f) ? g : 0.0f;
    return __fmul_rn(__fmul_rn(r, r), u);
}
// One lane of silu_inplace_avx512's vector body (quantization.rs:243-272).
__device__ __forceinline__ float silu_poly(float g, float u) {
    const float inv_ln2 = 1.44269504088896341f, ln2 = 0.693147180559945309f;
    const float hi = 88.3762626647949f, lo = -88.3762626647949f;
    float x = __fsub_rn(0.0f, g);
    x = (x < hi) ? x : hi;  // MINPS: second operand unless x < hi (NaN -> hi)
    x = (x > lo) ? x : lo;  // MAXPS
    const float fx = __fmul_rn(x, inv_ln2);
    const float n_f = __builtin_rintf(fx);
    const float t = __fsub_rn(x, __fmul_rn(n_f, ln2));
    float e = __fmaf_rn(1.0f / 24.0f, t, 1.0f / 6.0f);
    e = __fmaf_rn(e, t, 0.5f);
    e = __fmaf_rn(e, t, 1.0f);
    e = __fmaf_rn(e, t, 1.0f);
    const uint32_t bits = ((uint32_t)(int)n_f + 127u) << 23;
    const float exp_x = __fmul_rn(e, __uint_as_float(bits));
    const float sig = __fdiv_rn(1.0f, __fadd_rn(1.0f, exp_x));
    return __fmul_rn(__fmul_rn(g, sig), u);
}

__device__ __forceinline__ float apply_act(int act, float g, float u, bool main_lane) {
    switch (act) {
        case XT_ACT_SILU_INPLACE_AVX512:
            return main_lane ? silu_poly(g, u) : silu_scalar(g, u);
        case XT_ACT_SILU_INPLACE_SCALAR:
            return silu_scalar(g, u);
        case XT_ACT_SILU_MUL:
            return silu_div(g, u);
        case kActIdentity:
            return g;
        default:
            return relu2_mul(g, u);
    }
}

constexpr uint32_t kGrid = 1u << 24;                 // grid points per binade

// Wave-wide data movement with DPP (gfx9 encodings): row_shr:n = 0x110 + n
// shifts within rows of 16 lanes, row_bcast:15 / row_bcast:31 = 0x142 / 0x143
// broadcast lane 15 / 31 into the following rows, wave_shr:1 = 0x138 and
// wave_shl:1 = 0x130 shift across the whole wave.  Lanes without a source
// (or outside ROW_MASK) receive 0.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xf, false);
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint64_t dpp64(uint64_t v) {
    const uint32_t lo = dpp32<CTRL, ROW_MASK>((uint32_t)v);
    const uint32_t hi = dpp32<CTRL, ROW_MASK>((uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

// Inclusive wave scans (Hillis-Steele in rows of 16, then row broadcasts).
__device__ __forceinline__ uint64_t wave_scan_add(uint64_t v) {
    v += dpp64<0x111, 0xf>(v);
    v += dpp64<0x112, 0xf>(v);
    v += dpp64<0x114, 0xf>(v);
    v += dpp64<0x118, 0xf>(v);
    v += dpp64<0x142, 0xa>(v);
    v += dpp64<0x143, 0xc>(v);
    return v;
}
__device__ __forceinline__ uint32_t wave_scan_add(uint32_t v) {
    v += dpp32<0x111, 0xf>(v);
    v += dpp32<0x112, 0xf>(v);
    v += dpp32<0x114, 0xf>(v);
    v += dpp32<0x118, 0xf>(v);
    v += dpp32<0x142, 0xa>(v);
    v += dpp32<0x143, 0xc>(v);
    return v;
}
// Wave maximum of non-negative floats (0 is the identity), in every lane.
__device__ __forceinline__ float wave_max_nonneg(float v) {
    v = fmaxf(v, __uint_as_float(dpp32<0x111, 0xf>(__float_as_uint(v))));
    v = fmaxf(v, __uint_as_float(dpp32<0x112, 0xf>(__float_as_uint(v))));
    v = fmaxf(v, __uint_as_float(dpp32<0x114, 0xf>(__float_as_uint(v))));
    v = fmaxf(v, __uint_as_float(dpp32<0x118, 0xf>(__float_as_uint(v))));
    v = fmaxf(v, __uint_as_float(dpp32<0x142, 0xa>(__float_as_uint(v))));
    v = fmaxf(v, __uint_as_float(dpp32<0x143, 0xc>(__float_as_uint(v))));
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), 63));
}
__device__ __forceinline__ int wave_sum_int(int v) {
    const uint32_t s = wave_scan_add((uint32_t)v);
    return (int)__builtin_amdgcn_readlane(s, 63);
}
template <typename T>
__device__ __forceinline__ T lane_read(T v, int k) {
    if constexpr (sizeof(T) == 8) {
        const uint64_t b = __builtin_bit_cast(uint64_t, v);
        const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, k);
        const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), k);
        return __builtin_bit_cast(T, ((uint64_t)hi << 32) | lo);
    } else {
        return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(uint32_t, v), k));
    }
}

// Integer increment of adding t (finite, >= 0) to a running sum on the grid
// u = 2^(b-23): q = floor(t / u) (capped at 2^24), r = 0 below half, 1 at an
// exact half, 2 above.
__device__ __forceinline__ void grid_split(float t, int b, uint32_t* q, int* r) {
    const uint32_t bits = __float_as_uint(t);
    const uint32_t ef = (bits >> 23) & 0xffu;
    const uint32_t m = ef ? ((bits & 0x7fffffu) | 0x800000u) : (bits & 0x7fffffu);
    const int et = ef ? (int)ef - 150 : -149;
    const int shift = (b - 23) - et;
    // shift <= 0: t is a multiple of u (q = m << -shift, capped at 2^24)
    // (m >= 2^23 here: shifted by 8 or more it is past the cap)
    const int ls = min(-shift, 8);
    const uint32_t qup = min(m << max(ls, 0), kGrid);
    // shift > 0: m < 2^24, so shifts of 25 or more leave q = 0, remainder m
    const int sc = min(max(shift, 1), 25);
    const uint32_t qdn = m >> sc;
    const uint32_t rem = m & ((1u << sc) - 1u), half = 1u << (sc - 1);
    const int rdn = rem < half ? 0 : (rem == half ? 1 : 2);
    *q = shift <= 0 ? (m ? qup : 0u) : qdn;
    *r = shift <= 0 ? 0 : rdn;
}

__device__ __forceinline__ float wave_scan_addf(float v) {
    v = __fadd_rn(v, __uint_as_float(dpp32<0x111, 0xf>(__float_as_uint(v))));
    v = __fadd_rn(v, __uint_as_float(dpp32<0x112, 0xf>(__float_as_uint(v))));
    v = __fadd_rn(v, __uint_as_float(dpp32<0x114, 0xf>(__float_as_uint(v))));
    v = __fadd_rn(v, __uint_as_float(dpp32<0x118, 0xf>(__float_as_uint(v))));
    v = __fadd_rn(v, __uint_as_float(dpp32<0x142, 0xa>(__float_as_uint(v))));
    v = __fadd_rn(v, __uint_as_float(dpp32<0x143, 0xc>(__float_as_uint(v))));
    return v;
}
// Binade of a float >= 0 (subnormals and 0 in -126, infinity 128).
__device__ __forceinline__ int binade_f(float a) {
    const int e = (int)(__float_as_uint(a) >> 23);
    return e == 0 ? -126 : e - 127;
}

// Significand of s >= 0 on the grid of its binade (implicit bit included;
// for binade -126 the subnormal or smallest-normal encoding), and the float
// of significand T < 2^24 in binade b.
__device__ __forceinline__ int sig_binade(float s, uint32_t* S) {
    const uint32_t sbits = __float_as_uint(s);
    const int se = (int)(sbits >> 23);
    *S = (sbits & 0x7fffffu) | (se ? 0x800000u : 0u);
    return se == 0 ? -126 : se - 127;
}
__device__ __forceinline__ float from_grid(uint64_t T, int b) {
    return __uint_as_float(T >= 0x800000u ? ((uint32_t)(b + 127) << 23) | ((uint32_t)T & 0x7fffffu)
                                          : (uint32_t)T);  // b = -126, subnormal
}

// s + lt[j] + ... + lt[end - 1], each partial sum rounded to f32, by one
// whole wave (s is the same in every lane): 256 elements at a time (4
// consecutive ones per lane) are split on the grid of the running sum's
// binade and prefix-summed; the leading ones that are no tie and keep the sum
// inside the binade are added at once (exact integer addition on the grid),
// the next one with a real f32 add.
__device__ float seq_advance(float s, const float* lt, int j, int end) {
    const int lane = threadIdx.x & 63;
    s = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(s)));
    while (j < end) {
        uint32_t S;
        const int bs = sig_binade(s, &S);
        if (bs > 127) return s;  // infinity plus finite non-negative terms
        // lane l: elements j + 4 l .. j + 4 l + 3; local inclusive prefixes
        uint32_t pre[4];
        int kbad = 4;  // first element of the lane that is a tie or past `end`
        uint32_t acc = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int e = j + 4 * lane + k;
            uint32_t q = 0;
            int r = 1;  // past the end: treated as a stop
            if (e < end) grid_split(lt[e], bs, &q, &r);
            if (r == 1 && kbad == 4) kbad = k;
            acc += min(q + (r == 2 ? 1u : 0u), kGrid);
            pre[k] = acc;  // <= 4 * 2^24 per lane
        }
        // <= 256 * 2^24 = 2^32.  (Exactly 2^32 wraps to 0 in lane 63 only; then
        // the lane's exclusive prefix, at most 252 * 2^24, is right, and its
        // first element is a stop: S + lexcl + pre >= 2^24 in 64 bits.)
        const uint32_t lincl = wave_scan_add(acc);
        const uint32_t lexcl = lincl - acc;
        // first element (in order) that is a stop or leaves the binade
        int kfirst = kbad;
#pragma unroll
        for (int k = 3; k >= 0; --k)
            if ((uint64_t)S + lexcl + pre[k] >= kGrid) kfirst = min(kfirst, k);
        const uint64_t bad = __ballot(kfirst < 4);
        int m;  // elements added on the grid
        uint32_t pm = 0;
        if (bad) {
            const int L = (int)__builtin_ctzll(bad);
            const int kL = lane_read(kfirst, L);
            m = 4 * L + kL;
            if (m > 0) {
                // prefix through element m - 1
                uint32_t mine = 0;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (k == kL - 1) mine = lexcl + pre[k];
                pm = kL > 0 ? lane_read(mine, L) : lane_read(lincl, L - 1);
            }
        } else {
            m = 256;
            pm = lane_read(lincl, 63);
        }
        if (m > 0) {
            s = from_grid((uint64_t)S + pm, bs);
            j += m;
        }
        if (m < 256 && j < end) {
            s = __fadd_rn(s, lt[j]);
            ++j;
        }
        s = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(s)));
    }
    return s;
}

// Sequential float sum t[0] + t[1] + ... + t[n-1] (each partial sum rounded
// to f32, in index order) -- the order of rms_norm's sum of squares --
// computed by the whole workgroup.  Within one binade [2^b, 2^(b+1)) of the
// running sum, every f32 add is an integer add on the grid u = 2^(b-23):
// fl(s + t) = s + r, r = t rounded to a multiple of u, except when t lies
// half way between two multiples (a tie, whose rounding depends on the parity
// of s) or when the sum leaves the binade.  So:
//  1. thread j takes the E consecutive elements from j * E (E odd, so that
//     the threads' LDS reads fall on different banks), and a float prefix sum
//     predicts the binade at the start and the end of each thread's block;
//  2. a block is regular when both agree and none of its elements is a tie.
//     Rounding to the grid is one add and one subtract of 2^b, a tie one
//     subtract and one compare; the rounded elements add up exactly in f32;
//  3. one wave walks the other blocks in order with the running sum's bits
//     uniform: the regular blocks before one are a single integer add on the
//     bits if these lie in the run's precomputed range (the sum is in the
//     predicted binade and stays below its top), else seq_advance adds their
//     elements; the block's own elements are real f32 adds.
// The result never depends on the prediction being right, only the speed
// does.  `lt` holds t[0..n) (finite, >= 0) in LDS, `total` receives the float
// prefix sum of everything (NaN or infinite if an element or the sum is: then
// the caller decides).
//
// Per element 9 vector instructions, against about 45 when every element was
// split into grid increment and remainder with integer shifts.
template <int NT>
struct SeqSumLds {
    float wtot[NT / 64];
    uint64_t wgp[NT / 64];
    int wcnt[NT / 64];
    float res;
    int rec_blk[NT];       // irregular blocks in order
    int rec_b[NT];         // binade at their start
    uint64_t rec_gp[NT];   // grid increments of all regular blocks before them
};

template <int NT, int EB>
__device__ __forceinline__ float exact_seq_sum(int n, const float* lt, SeqSumLds<NT>& sl, float* total) {
    constexpr int NW = NT / 64;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int E = ((n + NT - 1) / NT) | 1;
    const int i0 = tid * E;
    const int cnt = max(0, min(E, n - i0));  // this thread's elements: [i0, i0 + cnt)
    float t[EB];
#pragma unroll
    for (int e = 0; e < EB; ++e) t[e] = e < cnt ? lt[i0 + e] : 0.0f;
    float acc = 0.0f;
#pragma unroll
    for (int e = 0; e < EB; ++e) acc = __fadd_rn(acc, t[e]);
    const float incl = wave_scan_addf(acc);
    const float excl = __uint_as_float(dpp32<0x138, 0xf>(__float_as_uint(incl)));  // wave_shr:1
    if (lane == 63) sl.wtot[w] = incl;
    __syncthreads();
    float woff = 0.0f, all = 0.0f;
#pragma unroll
    for (int j = 0; j < NW; ++j) {
        if (j == w) woff = all;
        all = __fadd_rn(all, sl.wtot[j]);
    }
    *total = all;
    if (!(all < __builtin_inff())) return 0.0f;  // uniform: every thread has the same sum
    const int b = binade_f(__fadd_rn(woff, excl)), bn = binade_f(__fadd_rn(woff, incl));
    // (every float is on the grid of binade -126: no rounding, no ties)
    const float top = b == -126 ? 0.0f : __uint_as_float((uint32_t)(b + 127) << 23);
    const float half = b == -126 ? -1.0f : __builtin_ldexpf(1.0f, b - 24);
    float R = 0.0f;
    bool irr = bn != b || tid == 0 || i0 + cnt == n;
#pragma unroll
    for (int e = 0; e < EB; ++e) {
        const float r = __fsub_rn(__fadd_rn(t[e], top), top);
        irr |= fabsf(__fsub_rn(t[e], r)) == half;
        R = __fadd_rn(R, r);
    }
    irr &= cnt > 0;
    // (R / u <= 2^24 where the block is used; anything larger fails the range)
    const uint32_t Q = irr ? 0u : (uint32_t)fminf(__builtin_ldexpf(R, 23 - b), 33554432.0f);
    const uint64_t gincl = wave_scan_add((uint64_t)Q);
    const uint64_t ballot = __ballot(irr);
    if (lane == 63) {
        sl.wgp[w] = gincl;
        sl.wcnt[w] = __builtin_popcountll(ballot);
    }
    __syncthreads();
    uint64_t gp = gincl;
    int rank = __builtin_popcountll(ballot & (((uint64_t)1 << lane) - 1));
    int nrec = 0;
#pragma unroll
    for (int j = 0; j < NW; ++j) {
        if (j < w) {
            gp += sl.wgp[j];
            rank += sl.wcnt[j];
        }
        nrec += sl.wcnt[j];
    }
    if (irr) {
        sl.rec_blk[rank] = tid;
        sl.rec_gp[rank] = gp;  // (own increment is 0)
        sl.rec_b[rank] = b;
    }
    __syncthreads();

    // The walk (wave 0).  Records are loaded 64 at a time, one per lane, with
    // everything that does not depend on the running sum: the range [lo, lim)
    // of running-sum bits for which the run's P increments are one integer add
    // on the bits (in binade b the bits are ((b + 127) << 23) + significand -
    // 2^23, or the significand itself for b = -126, so "sum in binade b and
    // sum + P below 2^(b+1)" is lo <= bits < hi - P).
    if (w == 0) {
        nrec = __builtin_amdgcn_readfirstlane(nrec);
        uint32_t sbits = 0;
        for (int k0 = 0; k0 < nrec; k0 += 64) {
            const int k = k0 + lane;
            int blk = 0, prev = -1;
            uint32_t lo = 0, lim = 0xffffffffu, P32 = 0;
            if (k < nrec) {
                blk = sl.rec_blk[k];
                prev = k > 0 ? sl.rec_blk[k - 1] : -1;
                if (prev + 1 < blk) {
                    const int rb = sl.rec_b[k];
                    const uint64_t P = sl.rec_gp[k] - (k > 0 ? sl.rec_gp[k - 1] : 0ull);
                    const uint32_t hi = (uint32_t)(rb + 128) << 23;
                    lo = rb == -126 ? 0u : (uint32_t)(rb + 127) << 23;
                    if (P >= (uint64_t)(hi - lo)) {
                        lo = 1u;  // empty range
                        lim = 0u;
                    } else {
                        lim = hi - (uint32_t)P;
                        P32 = (uint32_t)P;
                    }
                }
            }
            const int kn = min(64, nrec - k0);
            // element `lane` of block blk (0 past its end: adding it changes nothing)
            auto elements = [&](int kk) {
                const int i = lane_read(blk, kk) * E + lane;
                return lane < E && i < n ? lt[i] : 0.0f;
            };
            float x = elements(0);
            for (int kk = 0; kk < kn; ++kk) {
                const float xn = elements(min(kk + 1, kn - 1));
                const uint32_t klo = lane_read(lo, kk), klim = lane_read(lim, kk);
                const bool inr = sbits >= klo && sbits < klim;
                sbits = inr ? sbits + lane_read(P32, kk) : sbits;
                if (__builtin_expect(!inr, 0))
                    sbits = __float_as_uint(seq_advance(__uint_as_float(sbits), lt,
                                                        (lane_read(prev, kk) + 1) * E, lane_read(blk, kk) * E));
                float s = __uint_as_float(sbits);
#pragma unroll
                for (int e = 0; e < EB; ++e) s = __fadd_rn(s, lane_read(x, e));
                sbits = __builtin_amdgcn_readfirstlane(__float_as_uint(s));
                x = xn;
            }
        }
        if (lane == 0) sl.res = __uint_as_float(sbits);
    }
    __syncthreads();
    return sl.res;
}

// How a thread's elements lie in the row: pieces of four (rows of whole,
// 16-byte aligned pieces), single elements, or one single element in all.
constexpr int kPieces = 1, kSingles = 0, kOne = 2;

// One workgroup of NT threads per row; thread t holds C4 groups of four
// elements (kOne: one element) in registers from the load to the quantisation:
// pieces t, t + NT, ... or elements t, t + NT, ... (so that a wave's loads stay
// contiguous).  NORM: with RMSNorm.
//
// A row is bound by latency (the load, the walk of the sum, six barriers), so
// the width is what keeps enough rows in flight: see launch_mlp_mid.
// Measured, launch to launch, before (every element through integer grid
// increments, 1024 threads per row) and now: rms_norm of 2048 x 2560 37.5 ->
// 15.8 us, one row of 6912 11.1 -> 8.2, 512 x 6912 22.3 -> 13.8; silu_mul
// (no norm, f32 out) of 1024 x 8640 34.9 -> 24.6 (4.3 TB/s), the expf in
// double precision.
template <int ACT, int NT, int C4, int LIE, bool NORM>
__global__ __launch_bounds__(NT) void mid_kernel(const MidArgs a) {
    extern __shared__ __align__(16) float lt[];
    __shared__ float sm_f[NT / 64];
    constexpr bool VEC = LIE == kPieces;
    constexpr int G = LIE == kOne ? 1 : 4;  // elements per group
    static_assert(LIE != kOne || (C4 == 1 && !NORM), "one element per thread");
    const int m = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int n = a.n;
    const int nmain = (n / 16) * 16;
    const float* gr = a.gate + (size_t)m * a.ldg;
    const float* ur = a.up + (size_t)m * a.ldg;
    auto at = [&](int c, int e) { return VEC ? 4 * (c * NT + tid) + e : (G * c + e) * NT + tid; };
    // (elements past the row: 0)
    auto load4 = [&](const float* p, int c, float (&v)[G]) {
        if constexpr (VEC) {
            float4 x = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (at(c, 0) < n) x = *reinterpret_cast<const float4*>(p + at(c, 0));
            v[0] = x.x;
            v[1] = x.y;
            v[2] = x.z;
            v[3] = x.w;
        } else {
#pragma unroll
            for (int e = 0; e < G; ++e) v[e] = at(c, e) < n ? p[at(c, e)] : 0.0f;
        }
    };
    auto store4 = [&](float* p, int c, const float (&v)[G]) {
        if constexpr (VEC) {
            if (at(c, 0) < n) *reinterpret_cast<float4*>(p + at(c, 0)) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
            for (int e = 0; e < G; ++e)
                if (at(c, e) < n) p[at(c, e)] = v[e];
        }
    };
    float v[C4][G], nw[C4][G];
    {
        float g[C4][G], u[C4][G];
#pragma unroll
        for (int c = 0; c < C4; ++c) {
            load4(gr, c, g[c]);
            if constexpr (ACT != kActIdentity) load4(ur, c, u[c]);
        }
        if constexpr (NORM && C4 <= 4) {  // (fetched early where registers allow)
#pragma unroll
            for (int c = 0; c < C4; ++c) load4(a.norm_w, c, nw[c]);
        }
#pragma unroll
        for (int c = 0; c < C4; ++c)
#pragma unroll
            for (int e = 0; e < G; ++e) {
                v[c][e] = 0.0f;
                if (!VEC && (G * c + e) * NT >= n) continue;  // (uniform: short rows skip the code)
                v[c][e] = at(c, e) < n ? apply_act(ACT, g[c][e], ACT == kActIdentity ? 0.0f : u[c][e], at(c, e) < nmain)
                                       : 0.0f;
            }
    }
    if constexpr (NORM) {
        __shared__ SeqSumLds<NT> sl;
#pragma unroll
        for (int c = 0; c < C4; ++c) {
            const float t[4] = {__fmul_rn(v[c][0], v[c][0]), __fmul_rn(v[c][1], v[c][1]),
                                __fmul_rn(v[c][2], v[c][2]), __fmul_rn(v[c][3], v[c][3])};
            store4(lt, c, t);
        }
        __syncthreads();
        float total;
        float sum = exact_seq_sum<NT, 4 * C4 + 1>(n, lt, sl, &total);
        if (!(total < __builtin_inff())) {
            // NaN or infinity somewhere, or finite squares that overflow
            int f = 0;
            for (int i = tid; i < n; i += NT) f |= (lt[i] != lt[i] ? 1 : 0) | (__builtin_isinf(lt[i]) ? 2 : 0);
            const int wf = (__ballot(f & 1) ? 1 : 0) | (__ballot(f & 2) ? 2 : 0);
            if (lane == 0) sl.wcnt[w] = wf;
            __syncthreads();
            f = 0;
            for (int j = 0; j < NT / 64; ++j) f |= sl.wcnt[j];
            if (f == 0 && w == 0) {
                const float s = seq_advance(0.0f, lt, 0, n);
                if (lane == 0) sl.res = s;
            }
            __syncthreads();
            sum = (f & 1) ? __builtin_nanf("") : (f & 2) ? __builtin_inff() : sl.res;
        }
        // fast_attention_simd.rs:485-486.  sqrtf is correctly rounded on the
        // host; the hardware f32 square root is not, so take the correctly
        // rounded double root and round it once (exact: 53 >= 2*24 + 2).
        const float ms = __fadd_rn(__fdiv_rn(sum, (float)n), a.eps);
        const float rms = (float)__dsqrt_rn((double)ms);
        const float invr = __fdiv_rn(1.0f, rms);
#pragma unroll
        for (int c = 0; c < C4; ++c) {
            if constexpr (C4 > 4) load4(a.norm_w, c, nw[c]);
#pragma unroll
            for (int e = 0; e < G; ++e)
                if (at(c, e) < n) v[c][e] = __fmul_rn(__fmul_rn(v[c][e], invr), nw[c][e]);
        }
    }
    if (a.out) {
        float* orow = a.out + (size_t)m * a.ldo;
#pragma unroll
        for (int c = 0; c < C4; ++c) store4(orow, c, v[c]);
    }
    if (!a.q) return;
    float mx = 0.0f;
#pragma unroll
    for (int c = 0; c < C4; ++c)
#pragma unroll
        for (int e = 0; e < G; ++e) mx = fmaxf(mx, fabsf(v[c][e]));
    mx = wave_max_nonneg(mx);
    if (lane == 0) sm_f[w] = mx;
    __syncthreads();
    mx = 0.0f;
#pragma unroll
    for (int j = 0; j < NT / 64; ++j) mx = fmaxf(mx, sm_f[j]);
    const float scale = (mx > 0.0f) ? __fdiv_rn(127.0f, mx) : 1.0f;
    const float invs = (mx > 0.0f) ? __fdiv_rn(mx, 127.0f) : 1.0f;
    int8_t* qr = a.q + (size_t)m * a.ldq;
    // (the rounding mode is chosen once, so that only one quantiser's code
    // runs through the unrolled loop)
    auto quant_row = [&](auto mode_c) {
#pragma unroll
        for (int c = 0; c < C4; ++c) {
            int b[G];
#pragma unroll
            for (int e = 0; e < G; ++e) b[e] = quant_one(v[c][e], scale, decltype(mode_c)::value, at(c, e) < nmain) & 255;
            if constexpr (VEC) {
                if (at(c, 0) < n)
                    *reinterpret_cast<int*>(qr + at(c, 0)) = b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24);
            } else {
#pragma unroll
                for (int e = 0; e < G; ++e)
                    if (at(c, e) < n) qr[at(c, e)] = (int8_t)b[e];
            }
        }
    };
    if (a.mode == XT_QUANT_AVX512) quant_row(std::integral_constant<int, XT_QUANT_AVX512>{});
    else quant_row(std::integral_constant<int, XT_QUANT_SCALAR>{});
    for (int i = n + tid; i < a.ldq; i += NT) qr[i] = 0;
    if (tid == 0) a.inv[m] = invs;
}

int mid_max_cols() { return 16384; }

template <int NT, int C4, int LIE, bool NORM>
static hipError_t launch_mid_t(const MidArgs& a, int M, hipStream_t s) {
    const size_t lds = NORM ? (size_t)a.n * sizeof(float) : 0;
#define XT_MID(ACT_)                                                                          \
    case ACT_:                                                                                \
        hipLaunchKernelGGL((mid_kernel<ACT_, NT, C4, LIE, NORM>), dim3(M), dim3(NT), lds, s, a); \
        return hipGetLastError();
    switch (a.act) {
        XT_MID(XT_ACT_RELU2_MUL)
        XT_MID(XT_ACT_SILU_INPLACE_AVX512)
        XT_MID(XT_ACT_SILU_INPLACE_SCALAR)
        XT_MID(XT_ACT_SILU_MUL)
        case kActIdentity:  // (rms_norm alone)
            if constexpr (NORM) {
                hipLaunchKernelGGL((mid_kernel<kActIdentity, NT, C4, LIE, true>), dim3(M), dim3(NT), lds, s, a);
                return hipGetLastError();
            }
    }
#undef XT_MID
    return hipErrorInvalidValue;
}

hipError_t launch_mlp_mid(const MidArgs& a, int M, hipStream_t s) {
    if (M <= 0) return hipSuccess;
    if (a.n <= 0 || a.n > mid_max_cols()) return hipErrorInvalidValue;
    auto off = [](const void* p) { return ((uintptr_t)p & 15) != 0; };
    const bool vec = a.n % 4 == 0 && a.ldg % 4 == 0 && !off(a.gate) && (a.act == kActIdentity || !off(a.up)) &&
                     !off(a.norm_w) && (!a.out || (a.ldo % 4 == 0 && !off(a.out))) &&
                     (!a.q || (a.ldq % 4 == 0 && ((uintptr_t)a.q & 3) == 0));
    const int n4 = (a.n + 3) / 4;
#define XT_MIDT(NT_, C4_, LIE_, NORM_) \
    if (n4 <= NT_ * C4_) return launch_mid_t<NT_, C4_, LIE_, NORM_>(a, M, s);
    if (a.norm_w) {
        // Measured with 256 / 512 / 1024 threads per row, us: 1 x 2560 6.4 /
        // 6.6 / 7.4, 2048 x 2560 15.8 / 20.7 / 35.8 (narrow rows overlap one
        // another's walks); 1 x 6912 9.4 / 8.2 / 8.6, 512 x 6912 14.7 / 13.8 /
        // 17.5, 1024 x 8640 21.7 / 24.9 / 39.2 (long rows: the blocks of 256
        // threads get long, until there are more than two rows per CU).
        if (vec && (a.n <= 4096 || M > 512)) {
            XT_MIDT(256, 1, kPieces, true) XT_MIDT(256, 3, kPieces, true) XT_MIDT(256, 5, kPieces, true)
            XT_MIDT(256, 7, kPieces, true) XT_MIDT(256, 9, kPieces, true)
        }
        if (vec) { XT_MIDT(512, 4, kPieces, true) XT_MIDT(512, 8, kPieces, true) }
        XT_MIDT(512, 1, kSingles, true) XT_MIDT(512, 2, kSingles, true) XT_MIDT(512, 4, kSingles, true)
        XT_MIDT(512, 8, kSingles, true)
    } else {
        // One load, one reduction: wide rows (1 x 6912 7.7 / 5.8 / 4.5 us),
        // one element per thread where that is the row, as long as the rows
        // leave threads idle (one element each / four: 64 x 1003 2.13 / 2.34,
        // 300 x 64 2.03 / 2.53, 512 x 512 2.26 / 2.78, but 1024 x 1024 4.05 /
        // 3.66 and 4096 x 512 7.7 / 7.1; rows of 256 take it at any number,
        // 4096 x 256 3.87 / 4.45); then a piece per thread of 256 (2048 x 1024
        // 6.3 / 7.4 / 8.3 with 256 / 512 / 1024 threads), and fewer threads
        // again at more than two pieces per thread of 1024 (1024 x 8640 25.9 /
        // 24.6 / 27.0).
        if (a.n <= 256) return launch_mid_t<256, 1, kOne, false>(a, M, s);
        if (a.n <= 512 && M <= 512) return launch_mid_t<512, 1, kOne, false>(a, M, s);
        if (a.n <= 1024 && M <= 256) return launch_mid_t<1024, 1, kOne, false>(a, M, s);
        if (a.n <= 1024) {
            if (vec) { XT_MIDT(256, 1, kPieces, false) }
            XT_MIDT(256, 1, kSingles, false)
        }
        if (vec && a.n > 1024) {
            if (a.n > 8192 && M >= 512) { XT_MIDT(512, 5, kPieces, false) XT_MIDT(512, 8, kPieces, false) }
            XT_MIDT(1024, 1, kPieces, false) XT_MIDT(1024, 2, kPieces, false) XT_MIDT(1024, 4, kPieces, false)
        }
        XT_MIDT(1024, 1, kSingles, false) XT_MIDT(1024, 2, kSingles, false) XT_MIDT(1024, 4, kSingles, false)
    }
#undef XT_MIDT
    return hipErrorInvalidValue;
}

}  // namespace xt
