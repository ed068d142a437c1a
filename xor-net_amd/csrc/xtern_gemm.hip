// xtern prefill GEMM for many rows (gfx950): ternary tiles x i8 rows on
// v_mfma_i32_32x32x32_i8, the whole K in one workgroup.
//
// Reference behaviour: TernaryLinear::forward over several tokens
// (src/bit1_58/layers.rs:298-313), epilogue :306.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/xtern.h"
#include "xtern_device.h"
#include "xtern_internal.h"

namespace xt {

namespace {

typedef int v16i __attribute__((ext_vector_type(16)));

__device__ __forceinline__ v16i mfma32(v4i a, v4i b, v16i c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
}

// Sixteen 2-bit codes -> the sixteen NEGATED weights.  v_perm_b32's selector
// bytes 0..3 pick a byte of its second operand, 4..7 one of its first, 8 the
// replicated sign of the second's byte 1, 12 zero; a code field left in bits
// 2-3 of its byte is thus a selector as it is (0, 4, 8, 12), so only one shift
// is needed for the four fields: 9 VALU instructions per 16 weights (11 with
// a shift per field, which the signed decode of the other kernels takes).
__device__ __forceinline__ v4i decode_neg(int x) {
    const unsigned u = (unsigned)x, v = u >> 4;
    v4i b;
    b[0] = (int)__builtin_amdgcn_perm(0u, 0x00ff0001u, u & 0x03030303u);  // 0,1,2,3 -> 1, 0, -1, 0
    b[1] = (int)__builtin_amdgcn_perm(0u, 0x00008001u, u & 0x0c0c0c0cu);  // 0,4,8,12 -> 1, 0, -1, 0
    b[2] = (int)__builtin_amdgcn_perm(0u, 0x00ff0001u, v & 0x03030303u);
    b[3] = (int)__builtin_amdgcn_perm(0u, 0x00008001u, v & 0x0c0c0c0cu);
    return b;
}

// A buffer of `bytes` bytes at p (uniform); loads past it return zero.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
// 16 bytes per lane from buffer b (at lane offset + uniform offset) straight
// into LDS; the wave's 64 lanes fill 1 KiB at `dst` in lane order.
__device__ __forceinline__ void copy_lds16(__amdgpu_buffer_rsrc_t b, unsigned lane_off, unsigned off,
                                           uint8_t* dst) {
#if __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_raw_ptr_buffer_load_lds(b, (__attribute__((address_space(3))) void*)dst, 16,
                                             (int)lane_off, (int)off, 0, 0);
#endif
}
// Wait until at most VM of the wave's vector-memory operations are
// outstanding and its LDS reads are done, then meet the workgroup.
template <int VM>
__device__ __forceinline__ void wait_copies() {
    static_assert(VM >= 0 && VM < 64, "vmcnt is six bits");
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4));  // lgkmcnt 0
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
}

// Instruction order of one k-step: B times an MFMA followed by its share of
// the R fragment reads, the V loads and VALU vector instructions, which run
// while the matrix core works.
template <int I, int B, int R, int V, int VALU>
__device__ __forceinline__ void interleave() {
    if constexpr (I < B) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if constexpr ((R + B - 1 - I) / B > 0) __builtin_amdgcn_sched_group_barrier(0x100, (R + B - 1 - I) / B, 0);
        if constexpr ((V + B - 1 - I) / B > 0) __builtin_amdgcn_sched_group_barrier(0x010, (V + B - 1 - I) / B, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, VALU, 0);
        interleave<I + 1, B, R, V, VALU>();
    }
}

// The projection of workgroup column bx (scalar loads from the argument
// segment, as in xtern_kernels.hip).
typedef const __attribute__((address_space(4))) MMArgs* KArgPtr;

}  // namespace

// Workgroup tile: 32 MW tokens x 32 NW W output rows over all of K, W waves
// side by side along the rows; a wave multiplies all of the tile's tokens with
// its 32 NW rows (MW x NW accumulator blocks of 32 x 32).
//
// What bounds it: on long prompts the matrix cores at the clock they are left
// (1.8 to 1.95 GHz under this load; 60 to 66 % of the cycles have an MFMA in
// flight, by the counter that the cycles are taken from),
// on shapes of one workgroup per CU the issue of one wave per SIMD: 9 (Pack5
// 24) decode instructions per weight block and k-step next to 32 cycles per
// MFMA.  So:
//  * Activations go through LDS (every wave reads all of them); weights do
//    not: a wave's 2-bit tiles are a quarter of its activation bytes and no
//    other wave uses them, so each lane loads its own 16-byte tile slots (one
//    slot holds four k-steps of 32 columns) and decodes them in registers,
//    once for all 32 MW tokens.
//  * Activation chunks are copied straight from memory to LDS (no registers),
//    D chunks ahead, with one barrier per chunk.  The D buffers are separate
//    arrays and the waits are builtins: the compiler then sees that reading
//    one buffer does not depend on copies into the others, and adds no waits
//    of its own in the loop (one LDS array indexed by the chunk made it wait
//    for every copy in flight before each fragment read).
//  * LDS rows are unpadded (the copies fill them in lane order); instead each
//    lane copies a permuted 16-byte piece of its row, so that the 16 rows of a
//    fragment read fall on 16 different bank groups (no conflicts measured).
//  * Every k-step reads and decodes the next one's operands while its MFMAs
//    run, across chunk boundaries too: the last step of a chunk waits for the
//    next chunk and starts the loads of chunk c + D.
// The kernels it replaced (32 x 128 and 16 x 80 tiles) decoded every weight
// for 16 or 32 tokens only.  Measured, launch to launch: M = 4096, 4096 ->
// 14336 1094 -> 194 us (2.48 POP/s), M = 512, 2560 -> 13824 45 -> 21, 6912 ->
// 2560 32 -> 16; Pack5 M = 1024, 3200 -> 17280 226 -> 74, 8640 -> 3200 92 ->
// 37.  Two groups of waves taking alternate chunks (more waves per SIMD), and
// starting the workgroups that share operands at different chunks, changed
// nothing.
template <int FMT, int MW, int NW, int W, int D>
__global__ __launch_bounds__(64 * W, 2) void gemmw_kernel(const MMArgs a) {
    constexpr int STEPS = (FMT == XT_PACK5) ? 5 : 4;
    constexpr int CH = STEPS * 64;
    constexpr int MT = 32 * MW, NT = 32 * NW * W;
    constexpr int UNITS = MT * CH / 1024;       // 1 KiB direct-to-LDS copies per chunk
    constexpr int LPT = (UNITS + W - 1) / W;    // of them per wave
    __shared__ __align__(256) uint8_t lds0[MT * CH];
    __shared__ __align__(256) uint8_t lds1[MT * CH];
    __shared__ __align__(256) uint8_t lds2[D > 2 ? MT * CH : 16];
    __shared__ __align__(256) uint8_t lds3[D > 3 ? MT * CH : 16];
    __shared__ float sinv[MT];  // 1 / scale of the tile's tokens

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h = lane >> 5;
    const int r = lane & 31;

    KArgPtr ka = (KArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    const int np = ka->nproj, t1 = ka->proj[1].tile0, t2 = ka->proj[2].tile0, t3 = ka->proj[3].tile0;
    const int M = a.M, ldq = a.ldq, nch = a.nch;
    const int gx = a.gx, gy = (M + MT - 1) / MT;
    const int t = xcd_remap(blockIdx.x, gx * gy);
    const int grp = t / (8 * gx);
    const int gm = min(8, gy - 8 * grp);
    const int loc = t - 8 * gx * grp;
    const int bx = loc / gm;
    const int mbase = (8 * grp + loc - bx * gm) * MT;
    const int sel = ((np > 1) & (bx >= t1)) + ((np > 2) & (bx >= t2)) + ((np > 3) & (bx >= t3));
    const uint8_t* const tiles = ka->proj[sel].tiles;
    const int N = ka->proj[sel].N;
    const int obase = (bx - ka->proj[sel].tile0) * NT + wave * 32 * NW;  // the wave's first output row
    const int NG = (N + 15) >> 4;
    // The epilogue's operands are requested first: after the last MFMA they
    // were two memory round trips, and every store of a tile cut by M waited
    // for the one before (2560 -> 13824, M = 32 / 24: 8.12 / 8.84 -> 7.64 /
    // 7.68 us; 4096 -> 14336 with the quantiser, M = 500: 48.9 -> 44.9).
    const float* const ws = ka->proj[sel].ws;
    float* const y = ka->proj[sel].y;
    int32_t* const accout = ka->proj[sel].acc;
    float wsc[NW];
#pragma unroll
    for (int nb = 0; nb < NW; ++nb) wsc[nb] = ws[min(obase + 32 * nb + r, N - 1)];
    const float inv_of = a.inv[min(mbase + min((int)threadIdx.x, MT - 1), M - 1)];
    __asm__ volatile("" ::: "memory");

    // LDS unit (16 bytes) n of a chunk holds row n / (CH / 16), slot n % (CH /
    // 16); byte offsets of the pieces this lane copies.
    const __amdgpu_buffer_rsrc_t abuf =
        buffer_of(a.q + (size_t)mbase * ldq, (unsigned)min(MT, M - mbase) * (unsigned)ldq);
    const __amdgpu_buffer_rsrc_t wbuf = buffer_of(tiles, (unsigned)NG * (unsigned)nch * kTileBytes);
    unsigned goff[LPT];
    int unit[LPT];
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
        unit[i] = min(wave * LPT + i, UNITS - 1);  // (past the last: it once more)
        const int n = unit[i] * 64 + lane;
        const int row = n / (CH / 16), slot = n % (CH / 16);
        const int p = FMT == XT_PACK5 ? (slot ^ ((row >> 2) & 3)) : (slot ^ (row & 15));
        goff[i] = (unsigned)min(row, M - 1 - mbase) * (unsigned)ldq + 16u * p;
    }
    unsigned woff[NW];
#pragma unroll
    for (int nb = 0; nb < NW; ++nb) {
        const int G = min((obase >> 4) + 2 * nb + (r >> 4), NG - 1);
        woff[nb] = (unsigned)G * (unsigned)nch * kTileBytes + 256u * h + 16u * (r & 15);
    }

    v16i acc[MW][NW];
#pragma unroll
    for (int mb = 0; mb < MW; ++mb)
#pragma unroll
        for (int nb = 0; nb < NW; ++nb)
#pragma unroll
            for (int k = 0; k < 16; ++k) acc[mb][nb][k] = 0;

    v4i wv[D][NW][2];
    auto load_a = [&](int c, uint8_t* dst) {
        const unsigned off = (unsigned)min(c, nch - 1) * CH;
#pragma unroll
        for (int i = 0; i < LPT; ++i) copy_lds16(abuf, goff[i], off, dst + unit[i] * 1024);
    };
    auto load_w = [&](int c, v4i (&w)[NW][2]) {
        const unsigned off = (unsigned)min(c, nch - 1) * kTileBytes;
#pragma unroll
        for (int nb = 0; nb < NW; ++nb)
#pragma unroll
            for (int L = 0; L < 2; ++L)
                w[nb][L] = __builtin_amdgcn_raw_buffer_load_b128(wbuf, (int)(woff[nb] + 512u * L), (int)off, 0);
    };
    const unsigned fr = FMT == XT_PACK5 ? (unsigned)(r * CH) : (unsigned)(r * CH + 16 * (h ^ (r & 15)));
    auto read_f = [&](const uint8_t* src, int L, int s, v4i (&av)[MW]) {
        const unsigned fo = FMT == XT_PACK5 ? fr + 64u * s + 16u * ((2 * L + h) ^ ((r >> 2) & 3))
                                            : fr ^ (64u * s + 32u * L);
#pragma unroll
        for (int mb = 0; mb < MW; ++mb)
            av[mb] = *reinterpret_cast<const v4i*>(src + fo + mb * 32 * CH);
    };
    // Loads of chunk c, weights first (wait_copies counts them in this order).
    auto start = [&](int c, uint8_t* dst, v4i (&w)[NW][2]) {
        load_w(c, w);
        __asm__ volatile("" ::: "memory");
        load_a(c, dst);
        __asm__ volatile("" ::: "memory");
    };
    v4i av[2][MW], bv[2][NW];
    int E[NW][4], O[NW][4];
    auto decode = [&](int k, const v4i (&w)[NW][2], v4i (&b)[NW]) {
        const int L = k / STEPS, s = k % STEPS;
#pragma unroll
        for (int nb = 0; nb < NW; ++nb) {
            if constexpr (FMT == XT_PACK5) {
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    if (s == 0) {
                        E[nb][d] = w[nb][L][d] & 0x00ff00ff;
                        O[nb][d] = ((unsigned)w[nb][L][d] >> 8) & 0x00ff00ff;
                    }
                    const int pE = E[nb][d] * 3, pO = O[nb][d] * 3;
                    // the trits are selectors of the sign table as they are
                    b[nb][d] = (int)__builtin_amdgcn_perm(
                        0u, 0x00ff0001u, __builtin_amdgcn_perm((unsigned)pO, (unsigned)pE, 0x07030501u));
                    E[nb][d] = pE & 0x00ff00ff;
                    O[nb][d] = pO & 0x00ff00ff;
                }
            } else {
                b[nb] = decode_neg(w[nb][L][s]);
            }
        }
    };
    // Chunk c from its LDS buffer `src` and weights w; src2 / w2: the next
    // chunk's.  In every k-step the next one's fragments are read and its
    // weights decoded between the MFMAs; the last step of a chunk first waits
    // for the next chunk and starts the loads of chunk c + D into the buffer
    // and registers that chunk c no longer needs.  T >= 0: one of the last
    // chunks, T of them before it, with no loads left to start: the wait must
    // not count on any (weights that no later chunk multiplies are not even
    // loaded), and of the loads in flight it counts the copies only.
    auto step = [&](auto tail, int c, uint8_t* src, v4i (&w)[NW][2], const uint8_t* src2, v4i (&w2)[NW][2]) {
        constexpr int T = decltype(tail)::value;
        constexpr int B = MW * NW, VALU = (FMT == XT_PACK5 ? 24 : 9) * NW, VM = LPT + 2 * NW;
        constexpr bool more = T < D - 2;  // (T = D - 2: certainly the last)
#pragma unroll
        for (int k = 0; k < 2 * STEPS; ++k) {
            const bool last = k + 1 == 2 * STEPS;
            __builtin_amdgcn_sched_barrier(0);
            if (!last) {
                read_f(src, (k + 1) / STEPS, (k + 1) % STEPS, av[(k + 1) & 1]);
                decode(k + 1, w, bv[(k + 1) & 1]);
            } else if constexpr (more) {
                // (the loads of chunks c + 2 .. c + D - 1 - T may be in flight)
                if constexpr (T < 0) wait_copies<(D - 2) * VM>();
                else wait_copies<(D - 2 - T) * LPT>();
                __builtin_amdgcn_sched_barrier(0);
                read_f(src2, 0, 0, av[0]);
                if constexpr (T < 0) start(c + D, src, w);
                decode(0, w2, bv[0]);
            }
#pragma unroll
            for (int mb = 0; mb < MW; ++mb)
#pragma unroll
                for (int nb = 0; nb < NW; ++nb) acc[mb][nb] = mfma32(av[k & 1][mb], bv[k & 1][nb], acc[mb][nb]);
            if constexpr (B == 8 && T < 0) if (last) interleave<0, B, MW, VM, (VALU + B - 1) / B + 4>();
            if constexpr (B == 8) if (!last) interleave<0, B, MW, 0, (VALU + B - 1) / B>();
        }
    };
    start(0, lds0, wv[0]);
    __builtin_amdgcn_sched_barrier(0);
    start(1, lds1, wv[1]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (D > 2) start(2, lds2, wv[2]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (D > 3) start(3, lds3, wv[3]);
    __builtin_amdgcn_sched_barrier(0);
    wait_copies<(D - 1) * (LPT + 2 * NW)>();
    __builtin_amdgcn_sched_barrier(0);
    static_assert(MT <= 64 * W, "one scale per thread");
    if ((int)threadIdx.x < MT) sinv[threadIdx.x] = inv_of;
    read_f(lds0, 0, 0, av[0]);
    decode(0, wv[0], bv[0]);
    int c = 0;
    constexpr std::integral_constant<int, -1> loop{};
    constexpr std::integral_constant<int, 0> tail0{};
    if constexpr (D == 2) {
        for (; c + 2 <= nch; c += 2) {
            step(loop, c, lds0, wv[0], lds1, wv[1]);
            step(loop, c + 1, lds1, wv[1], lds0, wv[0]);
        }
        if (c < nch) step(tail0, c, lds0, wv[0], lds1, wv[1]);
    } else if constexpr (D == 3) {
        for (; c + 3 <= nch; c += 3) {
            step(loop, c, lds0, wv[0], lds1, wv[1]);
            step(loop, c + 1, lds1, wv[1], lds2, wv[2]);
            step(loop, c + 2, lds2, wv[2], lds0, wv[0]);
        }
        if (c < nch) step(tail0, c, lds0, wv[0], lds1, wv[1]);
        if (c + 1 < nch) step(std::integral_constant<int, 1>{}, c + 1, lds1, wv[1], lds2, wv[2]);
    } else {
        for (; c + 4 <= nch; c += 4) {
            step(loop, c, lds0, wv[0], lds1, wv[1]);
            step(loop, c + 1, lds1, wv[1], lds2, wv[2]);
            step(loop, c + 2, lds2, wv[2], lds3, wv[3]);
            step(loop, c + 3, lds3, wv[3], lds0, wv[0]);
        }
        if (c < nch) step(tail0, c, lds0, wv[0], lds1, wv[1]);
        if (c + 1 < nch) step(std::integral_constant<int, 1>{}, c + 1, lds1, wv[1], lds2, wv[2]);
        if (c + 2 < nch) step(std::integral_constant<int, 2>{}, c + 2, lds2, wv[2], lds3, wv[3]);
    }
    // (no copy into this workgroup's LDS outlives it)
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();

    // Register k of block (mb, nb): token 32 mb + 8 (k / 4) + 4 h + k % 4,
    // output row obase + 32 nb + r: each store of a wave writes two runs of
    // 128 bytes.
    auto write = [&](auto whole, auto with_acc) {
#pragma unroll
        for (int mb = 0; mb < MW; ++mb) {
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const int il = 32 * mb + 8 * (k >> 2) + 4 * h + (k & 3);
                if (!decltype(whole)::value && mbase + il >= M) continue;
                const float inv = sinv[il];
                const size_t at = (size_t)(mbase + il) * N + obase + r;
#pragma unroll
                for (int nb = 0; nb < NW; ++nb) {
                    if (!decltype(whole)::value && obase + 32 * nb + r >= N) continue;
                    const int d = -acc[mb][nb][k];
                    // layers.rs:306 — (dot as f32 * inv_scale) * w_scale, two roundings.
                    y[at + 32 * nb] = __fmul_rn(__fmul_rn((float)d, inv), wsc[nb]);
                    if (decltype(with_acc)::value) accout[at + 32 * nb] = d;
                }
            }
        }
    };
    if (accout)
        write(std::false_type{}, std::true_type{});
    else if (mbase + MT <= M && obase + 32 * NW <= N)
        write(std::true_type{}, std::false_type{});
    else
        write(std::false_type{}, std::false_type{});
}

// Compiled shapes: X(format, MW, NW, W, D).
#define XT_GW_SHAPES(X)                                                              \
    X(XT_PACK4, 4, 2, 4, 2) X(XT_PACK4, 2, 2, 4, 3) X(XT_PACK4, 2, 1, 4, 3)          \
    X(XT_PACK4, 1, 1, 4, 4) X(XT_PACK5, 4, 1, 8, 3) X(XT_PACK5, 4, 1, 4, 3)          \
    X(XT_PACK5, 2, 1, 4, 3) X(XT_PACK5, 1, 1, 4, 4)

bool gemmw_known(int fmt, int mw, int nw, int w) {
#define XT_GW(F_, MW_, NW_, W_, D_) \
    if ((fmt == XT_PACK5) == (F_ == XT_PACK5) && mw == MW_ && nw == NW_ && w == W_) return true;
    XT_GW_SHAPES(XT_GW)
#undef XT_GW
    return false;
}

hipError_t launch_gemmw(int fmt, int mw, int nw, int w, const MMArgs& a0, int ntiles, hipStream_t s) {
    MMArgs a = a0;
    a.gx = ntiles;
    const int gy = (a.M + 32 * mw - 1) / (32 * mw);
    if ((int64_t)ntiles * gy > 0x7fffffff) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(ntiles * gy));
#define XT_GW(F_, MW_, NW_, W_, D_)                                                            \
    if ((fmt == XT_PACK5) == (F_ == XT_PACK5) && mw == MW_ && nw == NW_ && w == W_) {           \
        hipLaunchKernelGGL((gemmw_kernel<F_, MW_, NW_, W_, D_>), grid, dim3(64 * W_), 0, s, a); \
        return hipGetLastError();                                                              \
    }
    XT_GW_SHAPES(XT_GW)
#undef XT_GW
    return hipErrorInvalidValue;
}

}  // namespace xt
