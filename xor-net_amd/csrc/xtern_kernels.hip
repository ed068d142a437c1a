// xtern HIP kernels for gfx950 (MI355X): activation quantiser and the
// ternary x i8 product on MFMA.
//
// Reference behaviour these kernels reproduce (paths relative to xor-net):
//   quantize_f32_to_i8          src/bit1_58/quantization.rs:95-195
//   ternary_dot_product_pack4   src/bit1_58/simd.rs:256-382
//   ternary_dot_product_pack5   src/bit1_58/simd.rs:384-414
//   TernaryLinear::forward      src/bit1_58/layers.rs:262-345 (epilogue :294)
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "../../include/xtern.h"
#include "xtern_internal.h"
#include "xtern_device.h"



namespace xt {

// One workgroup per row.  Pass 1: absmax (fmaxf ignores NaN; NaN inputs are
// off-contract).  Pass 2: quantise, write i8 (zero-filling [K, ldq)), and the
// exact i32 row sum the product kernels subtract.
__global__ __launch_bounds__(256) void quantize_kernel(const float* __restrict__ x, int64_t ldx,
                                                       int K, int8_t* __restrict__ q, int ldq,
                                                       float* __restrict__ inv,
                                                       int32_t* __restrict__ rowsum, int mode) {
    __shared__ float sm_f[4];
    __shared__ int sm_i[4];
    const int m = blockIdx.x;
    const float* xr = x + (size_t)m * ldx;
    int8_t* qr = q + (size_t)m * ldq;
    const bool vec = ((K & 3) == 0) && ((((uintptr_t)xr) & 15) == 0);

    float mx = 0.0f;
    if (vec) {
        const float4* x4 = reinterpret_cast<const float4*>(xr);
        for (int i = threadIdx.x; i < (K >> 2); i += 256) {
            const float4 v = x4[i];
            mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        }
    } else {
        for (int k = threadIdx.x; k < K; k += 256) mx = fmaxf(mx, fabsf(xr[k]));
    }
    mx = block_reduce(mx, MaxOp(), sm_f);
    const float scale = (mx > 0.0f) ? __fdiv_rn(127.0f, mx) : 1.0f;
    const float invs = (mx > 0.0f) ? __fdiv_rn(mx, 127.0f) : 1.0f;
    const int kmain = (K / 16) * 16;

    int sum = 0;
    if (vec && (ldq & 3) == 0 && ((((uintptr_t)qr) & 3) == 0)) {
        const float4* x4 = reinterpret_cast<const float4*>(xr);
        for (int i = threadIdx.x; i < (ldq >> 2); i += 256) {
            int b[4] = {0, 0, 0, 0};
            if (4 * i < K) {
                const float4 v = x4[i];
                const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int t = 0; t < 4; ++t) b[t] = quant_one(e[t], scale, mode, 4 * i + t < kmain);
            }
            sum += b[0] + b[1] + b[2] + b[3];
            const uint32_t packed = (uint32_t)(b[0] & 255) | ((uint32_t)(b[1] & 255) << 8) |
                                    ((uint32_t)(b[2] & 255) << 16) | ((uint32_t)(b[3] & 255) << 24);
            reinterpret_cast<uint32_t*>(qr)[i] = packed;
        }
    } else {
        for (int k = threadIdx.x; k < ldq; k += 256) {
            const int v = (k < K) ? quant_one(xr[k], scale, mode, k < kmain) : 0;
            qr[k] = (int8_t)v;
            sum += v;
        }
    }
    sum = block_reduce(sum, AddOp(), sm_i);
    if (threadIdx.x == 0) {
        inv[m] = invs;
        if (rowsum) rowsum[m] = sum;
    }
}

// Single-pass variant for K <= 4 * NT * NV with 16-byte aligned rows: each
// thread keeps its NV float4 of the row in registers between the absmax
// reduction and the quantisation, so the row is read from memory once.
// NT = 1024 for long rows (more loads in flight per row).
template <int NV, int NT>
__global__ __launch_bounds__(NT) void quantize_reg_kernel(const float* __restrict__ x, int64_t ldx,
                                                          int K, int8_t* __restrict__ q, int ldq,
                                                          float* __restrict__ inv,
                                                          int32_t* __restrict__ rowsum, int mode) {
    __shared__ float sm_f[NT / 64];
    __shared__ int sm_i[NT / 64];
    const int m = blockIdx.x;
    const float4* x4 = reinterpret_cast<const float4*>(x + (size_t)m * ldx);
    uint32_t* q4 = reinterpret_cast<uint32_t*>(q + (size_t)m * ldq);
    const int K4 = K >> 2;  // >= 1 (the launcher sends K < 4 elsewhere)
    // (every argument is consumed here, so all of them arrive in one round of
    // scalar loads ahead of the row load)
    asm volatile("" ::"s"(x), "s"(ldx), "s"(K), "s"(q), "s"(ldq), "s"(inv), "s"(rowsum), "s"(mode));
    float4 v[NV];
    float mx = 0.0f;
    // unconditional loads at clamped pieces, zeroed afterwards
#pragma unroll
    for (int u = 0; u < NV; ++u) v[u] = x4[min((int)threadIdx.x + u * NT, K4 - 1)];
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = threadIdx.x + u * NT;
        if (i >= K4) v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w))));
    }
    mx = block_reduce<NT / 64>(mx, MaxOp(), sm_f);
    const float scale = (mx > 0.0f) ? __fdiv_rn(127.0f, mx) : 1.0f;
    const float invs = (mx > 0.0f) ? __fdiv_rn(mx, 127.0f) : 1.0f;
    const int kmain = (K / 16) * 16;
    int sum = 0;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = threadIdx.x + u * NT;
        if (i >= K4) continue;
        const float e[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
        int b[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) b[t] = quant_one(e[t], scale, mode, 4 * i + t < kmain);
        sum += b[0] + b[1] + b[2] + b[3];
        q4[i] = (uint32_t)(b[0] & 255) | ((uint32_t)(b[1] & 255) << 8) |
                ((uint32_t)(b[2] & 255) << 16) | ((uint32_t)(b[3] & 255) << 24);
    }
    for (int i = K4 + threadIdx.x; i < (ldq >> 2); i += NT) q4[i] = 0u;  // padding
    if (rowsum) sum = block_reduce<NT / 64>(sum, AddOp(), sm_i);  // uniform: skipped when unused
    if (threadIdx.x == 0) {
        inv[m] = invs;
        if (rowsum) rowsum[m] = sum;
    }
}

// Row sums of caller-provided i8 activations, optionally copying them into a
// zero-padded buffer with a 16-byte aligned stride.
__global__ __launch_bounds__(256) void rowsum_kernel(const int8_t* __restrict__ qin, int64_t ldin,
                                                     int K, int8_t* __restrict__ qout, int ldout,
                                                     int32_t* __restrict__ rowsum) {
    __shared__ int sm_i[4];
    const int m = blockIdx.x;
    const int8_t* r = qin + (size_t)m * ldin;
    int sum = 0;
    const int lim = qout ? ldout : K;
    for (int k = threadIdx.x; k < lim; k += 256) {
        const int v = (k < K) ? (int)r[k] : 0;
        sum += v;
        if (qout) qout[(size_t)m * ldout + k] = (int8_t)v;
    }
    sum = block_reduce(sum, AddOp(), sm_i);
    if (threadIdx.x == 0) rowsum[m] = sum;
}

// The same for rows of any length and 4-byte alignment (ldx, K or the buffers
// not multiples of 4): the pieces of four are loaded and stored at whatever
// alignment they have (gfx950 takes it), the last K % 4 elements one by one.
// quantize_kernel reads such a row twice, one element per lane and step:
// 37 x 1003 4.3 -> 3.3 us, 300 x 7001 15.2 -> 5.1, 2048 x 3203 14.8 -> 11.2.
typedef float uf4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t uu32 __attribute__((aligned(1)));
template <int NV, int NT>
__global__ __launch_bounds__(NT) void quantize_any_kernel(const float* __restrict__ x, int64_t ldx, int K,
                                                          int8_t* __restrict__ q, int ldq,
                                                          float* __restrict__ inv,
                                                          int32_t* __restrict__ rowsum, int mode) {
    __shared__ float sm_f[NT / 64];
    __shared__ int sm_i[NT / 64];
    const int m = blockIdx.x;
    const float* xr = x + (size_t)m * ldx;
    int8_t* qr = q + (size_t)m * ldq;
    const int K4 = K >> 2, rem = K & 3;  // K4 >= 1
    float v[NV][4], tail = 0.0f;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = min((int)threadIdx.x + u * NT, K4 - 1);
        const uf4 t = *reinterpret_cast<const uf4*>(xr + 4 * i);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[u][e] = t[e];
    }
    if ((int)threadIdx.x < rem) tail = xr[4 * K4 + threadIdx.x];
    float mx = fabsf(tail);
#pragma unroll
    for (int u = 0; u < NV; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) mx = fmaxf(mx, fabsf(v[u][e]));  // (a clamped piece: its own maximum again)
    mx = block_reduce<NT / 64>(mx, MaxOp(), sm_f);
    const float scale = (mx > 0.0f) ? __fdiv_rn(127.0f, mx) : 1.0f;
    const float invs = (mx > 0.0f) ? __fdiv_rn(mx, 127.0f) : 1.0f;
    const int kmain = (K / 16) * 16;
    int sum = 0;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = threadIdx.x + u * NT;
        if (i >= K4) continue;
        int b[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) b[t] = quant_one(v[u][t], scale, mode, 4 * i + t < kmain);
        sum += b[0] + b[1] + b[2] + b[3];
        *reinterpret_cast<uu32*>(qr + 4 * i) = (uint32_t)(b[0] & 255) | ((uint32_t)(b[1] & 255) << 8) |
                                               ((uint32_t)(b[2] & 255) << 16) | ((uint32_t)(b[3] & 255) << 24);
    }
    if ((int)threadIdx.x < rem) {  // (past the last 16 elements: the scalar tail's rounding)
        const int b = quant_one(tail, scale, mode, false);
        sum += b;
        qr[4 * K4 + threadIdx.x] = (int8_t)b;
    }
    for (int i = K + threadIdx.x; i < ldq; i += NT) qr[i] = 0;  // padding
    if (rowsum) sum = block_reduce<NT / 64>(sum, AddOp(), sm_i);  // uniform: skipped when unused
    if (threadIdx.x == 0) {
        inv[m] = invs;
        if (rowsum) rowsum[m] = sum;
    }
}

hipError_t launch_quantize(const float* x, int64_t ldx, int M, int K, int8_t* q, int ldq,
                           float* inv, int32_t* rowsum, int mode, hipStream_t s) {
    if (M <= 0) return hipSuccess;
    const bool aligned = (K % 4 == 0) && (ldx % 4 == 0) && (ldq % 4 == 0) &&
                         ((uintptr_t)x % 16 == 0) && ((uintptr_t)q % 4 == 0);
    if (aligned && K >= 4 && K <= 16384) {
#define XT_QREG(NV_, NT_)                                                                        \
    if (K <= 4 * NT_ * NV_) {                                                                    \
        hipLaunchKernelGGL((quantize_reg_kernel<NV_, NT_>), dim3(M), dim3(NT_), 0, s, x, ldx, K, q, \
                           ldq, inv, rowsum, mode);                                              \
        return hipGetLastError();                                                                \
    }
        XT_QREG(1, 256)
        XT_QREG(2, 256)
        XT_QREG(1, 1024)
        XT_QREG(2, 1024)
        XT_QREG(4, 1024)
#undef XT_QREG
    }
    if (K >= 4 && K <= 16384 && (uintptr_t)x % 4 == 0) {
#define XT_QANY(NV_, NT_)                                                                        \
    if (K / 4 <= NT_ * NV_) {                                                                    \
        hipLaunchKernelGGL((quantize_any_kernel<NV_, NT_>), dim3(M), dim3(NT_), 0, s, x, ldx, K, q, \
                           ldq, inv, rowsum, mode);                                              \
        return hipGetLastError();                                                                \
    }
        XT_QANY(1, 256)
        XT_QANY(2, 256)
        XT_QANY(1, 1024)
        XT_QANY(2, 1024)
        XT_QANY(4, 1024)
#undef XT_QANY
    }
    hipLaunchKernelGGL(quantize_kernel, dim3(M), dim3(256), 0, s, x, ldx, K, q, ldq, inv, rowsum,
                       mode);
    return hipGetLastError();
}

// Static scratch of the allocation-free entry point: device memory that the
// library never allocates at run time.  Each GPU holds its own copy; host
// code reaches it only through the address hipGetSymbolAddress returns for
// the current device (the array's name is a host-side stand-in).  Every call
// on one GPU shares it: calls that overlap on one GPU race.
constexpr size_t kScratchBytes = (size_t)8 << 20;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

hipError_t scratch_region(void** ptr, size_t* bytes) {
    static std::mutex mu;
    static void* addr[64] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(mu);
    if (!addr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        addr[dev] = p;
    }
    *ptr = addr[dev];
    *bytes = kScratchBytes;
    return hipSuccess;
}

hipError_t launch_rowsum(const int8_t* qin, int64_t ldin, int M, int K, int8_t* qout, int ldout,
                         int32_t* rowsum, hipStream_t s) {
    if (M <= 0) return hipSuccess;
    hipLaunchKernelGGL(rowsum_kernel, dim3(M), dim3(256), 0, s, qin, ldin, K, qout, ldout, rowsum);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Ternary x i8 product on MFMA
// ---------------------------------------------------------------------------

// The projection workgroup column bx belongs to, read through the kernel
// argument segment (scalar loads; the selected projection is one load at a
// computed offset -- selecting among by-value fields instead makes the
// compiler copy the arguments to scratch memory).
struct ProjView {
    const uint8_t* tiles;
    const float* ws;
    float* y;
    int32_t* acc;
    int N, tile0, col0;
};
typedef const __attribute__((address_space(4))) MMArgs* KArgPtr;
struct ProjBounds {
    int np, t0, t1, t2, t3;
};
// Read at kernel entry, in the same round of scalar loads as the grid size.
// proj[0].tile0 (always 0) is read in this round too: it shares the first
// argument line with proj[0]'s pointers, so that line is fetched beside the
// bounds and the selected projection's load (proj[0] in a single-projection
// launch) hits the scalar cache instead of waiting on a second cold line.
__device__ __forceinline__ ProjBounds proj_bounds() {
    KArgPtr ka = (KArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    return ProjBounds{ka->nproj, ka->proj[0].tile0, ka->proj[1].tile0, ka->proj[2].tile0,
                      ka->proj[3].tile0};
}
__device__ __forceinline__ ProjView select_proj(const ProjBounds& pb, int bx) {
    KArgPtr ka = (KArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    bx -= pb.t0;  // (tile0 of the first projection is 0)
    const int sel = ((pb.np > 1) & (bx >= pb.t1)) + ((pb.np > 2) & (bx >= pb.t2)) +
                    ((pb.np > 3) & (bx >= pb.t3));
    ProjView v;
    v.tiles = ka->proj[sel].tiles;
    v.ws = ka->proj[sel].ws;
    v.y = ka->proj[sel].y;
    v.acc = ka->proj[sel].acc;
    v.N = ka->proj[sel].N;
    v.tile0 = ka->proj[sel].tile0;
    v.col0 = ka->proj[sel].col0;
    return v;
}

// Workgroup (blockIdx.x, blockIdx.y, blockIdx.z) computes a (16*MB tokens) x
// (16*NB output rows) tile over chunk slice z of the reduction dimension.  Its
// WAVES waves take interleaved chunks of the slice and are summed through
// LDS.  Each wave loads PF chunks (weights and activations) before consuming
// any, so one HBM round trip covers PF chunks.  With gridDim.z > 1 the slices
// write their partial sums to planes of a workspace; the last workgroup to
// arrive at a tile (device-scope counter, release/acquire fences) adds the
// planes, runs the epilogue and clears the counter for the next call.
// OWN_ROWSUM (MB == 1): the activation row sums come from one extra MFMA per
// k-step against an all-ones B operand instead of the caller.
#ifndef XT_MM_SLICE
#define XT_MM_SLICE 1
#endif
template <int FMT, int MB, int NB, int WAVES, int PF, bool OWN_ROWSUM>
__global__ __launch_bounds__(WAVES * 64) void mm_kernel(const MMArgs a) {
    constexpr int STEPS = (FMT == XT_PACK5) ? 5 : 4;
    constexpr int CH = STEPS * 64;
    constexpr int NBLK = MB * NB;
    constexpr int NACC = NBLK + (OWN_ROWSUM ? 1 : 0);
    static_assert(!OWN_ROWSUM || MB == 1, "in-kernel row sums need MB == 1");
    __shared__ v4i red[WAVES][NACC][64];
    __shared__ int last_flag;
    // SLICE (one 16-token block, 2-bit tiles): each activation load covers
    // 4 token rows x 256 bytes, one distinct 16-byte piece per lane, instead
    // of 16 rows x 64 bytes (an instruction spanning 16 rows at the row
    // stride kept the address path stalled on translation); the pieces go
    // through a wave-private LDS slice (rows padded by one piece) and come
    // back as MFMA fragments.  No barrier: a wave's LDS accesses complete in
    // order.
    constexpr bool SLICE = XT_MM_SLICE && FMT != XT_PACK5 && MB == 1 &&
                           WAVES * NACC * 1024 + WAVES * PF * 16 * 17 * 16 <= 150 * 1024;
    __shared__ v4i aslice[WAVES][SLICE ? PF : 1][SLICE ? 16 * 17 : 1];

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int g = lane >> 4;
    const int j = lane & 15;

    // Which projection this workgroup belongs to (constant-index selects keep
    // the kernel-argument struct out of scratch memory).
    const int bx = blockIdx.x;
    const ProjView pv = select_proj(proj_bounds(), bx);
    const uint8_t* tiles = pv.tiles;
    const float* ws = pv.ws;
    float* y = pv.y;
    int32_t* accout = pv.acc;
    const int N = pv.N;
    const int tile0 = pv.tile0;
    const int col0 = pv.col0;
    const int ntile = bx - tile0;
    const int NG = (N + 15) >> 4;
    const int M = a.M;
    const int mbase = blockIdx.y * (16 * MB);
    const int nch = a.nch;
    const int ldq = a.ldq;
    const int cbeg = blockIdx.z * a.cps;
    const int cend = min(nch, cbeg + a.cps);
    const int8_t* const qbase = a.q;
    // (consumed here, so the activation pointer and strides are loaded with
    // the projection's fields rather than in a third round inside the loop)
    asm volatile("" ::"s"(qbase), "s"(ldq), "s"(nch), "s"(M), "s"(cend), "s"(tiles));

    v4i acc[MB][NB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = v4i{0, 0, 0, 0};
    v4i accs = v4i{0, 0, 0, 0};
    const v4i ones = v4i{0x01010101, 0x01010101, 0x01010101, 0x01010101};
    const v4i zero = v4i{0, 0, 0, 0};

    for (int c0 = cbeg + wave; c0 < cend; c0 += WAVES * PF) {
        v4i wv[PF][NB];
        v4i av[PF][MB][STEPS];
#pragma unroll
        for (int pp = 0; pp < PF; ++pp) {
            const int c = c0 + pp * WAVES;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const int G = ntile * NB + nb;
                wv[pp][nb] = (c < cend && G < NG)
                                 ? ld_stream(tiles + ((size_t)(G * nch + c) * 64 + lane) * 16)
                                 : zero;
            }
            if constexpr (SLICE) {
                // (clamped rows and chunk: zeroed when read back)
                const int cc = min(c, cend - 1);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int row = min(mbase + 4 * u + (lane >> 4), M - 1);
                    av[pp][0][u] = ld_cached(qbase + (size_t)row * ldq + cc * CH + (lane & 15) * 16);
                }
            } else {
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                const int row = mbase + mb * 16 + j;
#pragma unroll
                for (int s = 0; s < STEPS; ++s)
                    av[pp][mb][s] = (c < cend && row < M)
                                        ? ld_cached(qbase + (size_t)row * ldq + c * CH + s * 64 + g * 16)
                                        : zero;
            }
            }
        }
        if constexpr (SLICE) {
            // rows 4u + lane / 16, piece lane % 16 -> the fragments of
            // lane (g, j): row j, pieces 4 s + g
#pragma unroll
            for (int pp = 0; pp < PF; ++pp)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    aslice[wave][pp][(4 * u + (lane >> 4)) * 17 + (lane & 15)] = av[pp][0][u];
            __asm__ volatile("" ::: "memory");
#pragma unroll
            for (int pp = 0; pp < PF; ++pp) {
                const bool live = c0 + pp * WAVES < cend && mbase + j < M;
#pragma unroll
                for (int s = 0; s < STEPS; ++s) {
                    const v4i v = aslice[wave][pp][j * 17 + 4 * s + g];
                    av[pp][0][s] = live ? v : zero;
                }
            }
        }
#pragma unroll
        for (int pp = 0; pp < PF; ++pp) {
            if (c0 + pp * WAVES >= cend) break;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                if constexpr (FMT == XT_PACK5) {
                    int E[4], O[4];
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        E[d] = wv[pp][nb][d] & 0x00ff00ff;
                        O[d] = ((unsigned)wv[pp][nb][d] >> 8) & 0x00ff00ff;
                    }
#pragma unroll
                    for (int s = 0; s < STEPS; ++s) {
                        v4i b;
#pragma unroll
                        for (int d = 0; d < 4; ++d) {
                            const int pE = E[d] * 3, pO = O[d] * 3;
                            b[d] = (int)__builtin_amdgcn_perm((unsigned)pO, (unsigned)pE, 0x07030501u);
                            E[d] = pE & 0x00ff00ff;
                            O[d] = pO & 0x00ff00ff;
                        }
#pragma unroll
                        for (int mb = 0; mb < MB; ++mb) acc[mb][nb] = mfma(av[pp][mb][s], b, acc[mb][nb]);
                        if constexpr (OWN_ROWSUM)
                            if (nb == 0) accs = mfma(av[pp][0][s], ones, accs);
                    }
                } else {
#pragma unroll
                    for (int s = 0; s < STEPS; ++s) {
                        const v4i b = decode4(wv[pp][nb][s]);
#pragma unroll
                        for (int mb = 0; mb < MB; ++mb) acc[mb][nb] = mfma(av[pp][mb][s], b, acc[mb][nb]);
                        if constexpr (OWN_ROWSUM)
                            if (nb == 0) accs = mfma(av[pp][0][s], ones, accs);
                    }
                }
            }
        }
    }

    // Reduction over the waves through LDS: every wave parks all its
    // accumulators, then wave w finishes blocks w, w + WAVES, ...
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) red[wave][mb * NB + nb][lane] = acc[mb][nb];
    if constexpr (OWN_ROWSUM) red[wave][NACC - 1][lane] = accs;
    __syncthreads();

    // OWN_ROWSUM: row sums of this slice's activations, laid out like the
    // accumulators (lane (g, j) register r belongs to token 4g + r).
    v4i rs = zero;
    if constexpr (OWN_ROWSUM) {
#pragma unroll
        for (int w = 0; w < WAVES; ++w) rs += red[w][NACC - 1][lane];
    }
    const bool split = gridDim.z > 1;

    if (split) {
        // Publish this slice's partial sums (code domain; an OWN_ROWSUM slice
        // has already subtracted its own share of the row sums) to plane z of
        // the workspace, then count arrivals at this tile.
        int32_t* plane = a.part + (size_t)blockIdx.z * a.M * a.ldp;
        for (int blk = wave; blk < NBLK; blk += WAVES) {
            const int mb = blk / NB, nb = blk % NB;
            v4i sum = zero;
#pragma unroll
            for (int w = 0; w < WAVES; ++w) sum += red[w][blk][lane];
            const int o = (ntile * NB + nb) * 16 + j;
            if (o >= N) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = mbase + mb * 16 + 4 * g + r;
                if (i >= M) continue;
                int ownr = 0;
                if constexpr (OWN_ROWSUM) ownr = rs[r];
                plane[(size_t)i * a.ldp + col0 + o] = sum[r] - ownr;
            }
        }
        __threadfence();  // release: the planes are visible device-wide
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned* c = a.cnt + (size_t)blockIdx.y * gridDim.x + blockIdx.x;
            const unsigned old = __hip_atomic_fetch_add(c, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
            last_flag = (old == gridDim.z - 1);
            if (last_flag) __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (!last_flag) return;
        __threadfence();  // acquire: see every other slice's plane
    }

    for (int blk = wave; blk < NBLK; blk += WAVES) {
        const int mb = blk / NB, nb = blk % NB;
        v4i sum = zero;
        if (!split) {
#pragma unroll
            for (int w = 0; w < WAVES; ++w) sum += red[w][blk][lane];
        }
        const int o = (ntile * NB + nb) * 16 + j;
        if (o >= N) continue;
        const float wscale = ws[o];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = mbase + mb * 16 + 4 * g + r;
            if (i >= M) continue;
            int d;
            if (split) {
                const size_t off = (size_t)i * a.ldp + col0 + o;
                const size_t plane_sz = (size_t)a.M * a.ldp;
                int tot = 0;
                for (unsigned z = 0; z < gridDim.z; ++z)
                    tot += __builtin_nontemporal_load(a.part + z * plane_sz + off);
                d = OWN_ROWSUM ? tot : tot - a.rowsum[i];
            } else {
                d = sum[r] - (OWN_ROWSUM ? rs[r] : a.rowsum[i]);
            }
            // layers.rs:294 — (dot as f32 * inv_scale) * w_scale, two roundings.
            y[(size_t)i * N + o] = __fmul_rn(__fmul_rn((float)d, a.inv[i]), wscale);
            if (accout) accout[(size_t)i * N + o] = d;
        }
    }
}

template <int FMT, int MB, int NB, int W, int PF, bool OWN>
static hipError_t launch_t(const MMArgs& a, int ntiles, int splitk, hipStream_t s) {
    dim3 grid(ntiles, (a.M + 16 * MB - 1) / (16 * MB), splitk);
    hipLaunchKernelGGL((mm_kernel<FMT, MB, NB, W, PF, OWN>), grid, dim3(W * 64), 0, s, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Decode GEMV (M <= 16): activations staged in LDS, all weights in flight
// ---------------------------------------------------------------------------
//
// Workgroup x owns the 16 output rows of row group x (or of the projection
// x falls in) over the full reduction dimension.  The M <= 16 activation
// rows go to LDS once ([chunk][step][g][token][16 B], only real tokens), so
// each wave keeps nothing but weights in registers: wave w loads chunks
// w, w + WAVES, ... (at most NCW each) before its first MFMA, one HBM round
// trip for the whole row group.  The exact row sums are taken while staging
// (v_dot4 against 1s, LDS atomics); the epilogue's scales are loaded at entry;
// waves are summed through LDS.
template <int FMT, int WAVES, int NCW>
__global__ __launch_bounds__(WAVES * 64) void gemv_kernel(const MMArgs a) {
    constexpr int STEPS = (FMT == XT_PACK5) ? 5 : 4;
    constexpr int CH = STEPS * 64;
    // 1 KiB tiles per chunk, and the weight code offset the activation row
    // sum removes: ternary codes are w + 1, Int4 codes q + 8, Int8 none.
    constexpr int TPC = (FMT == XT_INT8) ? 4 : (FMT == XT_INT4 ? 2 : 1);
    constexpr int OFF = (FMT == XT_INT8) ? 0 : (FMT == XT_INT4 ? 8 : 1);
    constexpr int SEGS = CH / 16;
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ v4i red[WAVES][64];
    __shared__ int rsum[16];
    __shared__ unsigned rmax[16];

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int g = lane >> 4;
    const int j = lane & 15;

    const int bx = blockIdx.x;
    const ProjView pv = select_proj(proj_bounds(), bx);
    const uint8_t* tiles = pv.tiles;
    const float* ws = pv.ws;
    float* y = pv.y;
    int32_t* accout = pv.acc;
    const int N = pv.N;
    const int tile0 = pv.tile0;
    const int G = bx - tile0;
    const int M = a.M;
    const int nch = a.nch;
    if (threadIdx.x < 16) rsum[threadIdx.x] = 0;

    // weights first: they come from HBM and take longest
    v4i wv[NCW][TPC];
#pragma unroll
    for (int t = 0; t < NCW; ++t) {
        const int c = wave + t * WAVES;
#pragma unroll
        for (int u = 0; u < TPC; ++u)
            wv[t][u] = c < nch ? ld_stream(tiles + (((size_t)(G * nch + c) * TPC + u) * 64 + lane) * 16)
                               : v4i{0, 0, 0, 0};
    }
    // epilogue operands, so no memory round trip is left after the MFMAs
    const int o = G * 16 + j;
    const float wscale = (wave == 0 && o < N) ? ws[o] : 0.0f;
    float invr[4];
    const bool fused = a.x != nullptr;
#pragma unroll
    for (int r = 0; r < 4; ++r) invr[r] = (!fused && wave == 0 && 4 * g + r < M) ? a.inv[4 * g + r] : 0.0f;
    if (threadIdx.x < 16) rmax[threadIdx.x] = 0u;
    __syncthreads();  // rsum / rmax cleared

    const int pieces = M * nch * SEGS;
    if (fused) {
        // Quantiser fused (quantization.rs:95-195, as quantize_kernel): every
        // piece (16 columns of one row) is read as f32, the row absmax is
        // gathered through LDS, then the piece is quantised into the stage.
        // The caller guarantees at most one piece per thread.
        const int p = threadIdx.x;
        const int m = p % M;
        const int seg = (p / M) % SEGS;
        const int c = p / (M * SEGS);
        const int col = c * CH + seg * 16;
        float f[16];
        float mx = 0.0f;
        if (p < pieces) {
            const float* xr = a.x + (size_t)m * a.ldx + col;
            if (col + 16 <= a.K && ((((uintptr_t)xr) & 15) == 0)) {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const float4 v = reinterpret_cast<const float4*>(xr)[t];
                    f[4 * t] = v.x;
                    f[4 * t + 1] = v.y;
                    f[4 * t + 2] = v.z;
                    f[4 * t + 3] = v.w;
                }
            } else {
#pragma unroll
                for (int t = 0; t < 16; ++t) f[t] = col + t < a.K ? xr[t] : 0.0f;
            }
#pragma unroll
            for (int t = 0; t < 16; ++t) mx = fmaxf(mx, fabsf(f[t]));  // NaN ignored
            atomicMax(&rmax[m], __float_as_uint(mx));  // non-negative floats order as ints
        }
        __syncthreads();
        if (p < pieces) {
            const float rmx = __uint_as_float(rmax[m]);
            const float scale = (rmx > 0.0f) ? __fdiv_rn(127.0f, rmx) : 1.0f;
            const int kmain = (a.K / 16) * 16;
            v4i v;
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                unsigned w4 = 0;
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int k = col + 4 * d + t;
                    const int b = k < a.K ? quant_one(f[4 * d + t], scale, a.mode, k < kmain) : 0;
                    w4 |= (unsigned)(b & 255) << (8 * t);
                }
                v[d] = (int)w4;
            }
            int part = 0;
#pragma unroll
            for (int d = 0; d < 4; ++d) part = __builtin_amdgcn_sdot4(v[d], 0x01010101, part, false);
            atomicAdd(&rsum[m], part);
            const int st = seg >> 2, gg = seg & 3;
            *reinterpret_cast<v4i*>(lds + ((((c * STEPS + st) * 4 + gg) * M + m) << 4)) = v;
        }
        __syncthreads();
        if (wave == 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float rmx = __uint_as_float(rmax[4 * g + r]);
                invr[r] = (4 * g + r < M) ? ((rmx > 0.0f) ? __fdiv_rn(rmx, 127.0f) : 1.0f) : 0.0f;
            }
        }
    } else {
        // activations -> LDS, with exact per-token byte sums (v_dot4 by 1s)
        for (int p = threadIdx.x; p < pieces; p += WAVES * 64) {
            const int m = p % M;
            const int seg = (p / M) % SEGS;
            const int c = p / (M * SEGS);
            const v4i v = ld_cached(a.q + (size_t)m * a.ldq + (size_t)c * CH + seg * 16);
            int part = 0;
#pragma unroll
            for (int d = 0; d < 4; ++d) part = __builtin_amdgcn_sdot4(v[d], 0x01010101, part, false);
            atomicAdd(&rsum[m], part);
            const int st = seg >> 2, gg = seg & 3;
            *reinterpret_cast<v4i*>(lds + ((((c * STEPS + st) * 4 + gg) * M + m) << 4)) = v;
        }
        __syncthreads();
    }

    // one accumulator per k-step: short dependent MFMA chains
    v4i acc[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) acc[s] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int t = 0; t < NCW; ++t) {
        const int c = wave + t * WAVES;
        if (c < nch) {
            if constexpr (FMT == XT_PACK5) {
                int E[4], O[4];
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    E[d] = wv[t][0][d] & 0x00ff00ff;
                    O[d] = ((unsigned)wv[t][0][d] >> 8) & 0x00ff00ff;
                }
#pragma unroll
                for (int s = 0; s < STEPS; ++s) {
                    v4i b;
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        const int pE = E[d] * 3, pO = O[d] * 3;
                        b[d] = (int)__builtin_amdgcn_perm((unsigned)pO, (unsigned)pE, 0x07030501u);
                        E[d] = pE & 0x00ff00ff;
                        O[d] = pO & 0x00ff00ff;
                    }
                    v4i av = v4i{0, 0, 0, 0};
                    if (j < M)
                        av = *reinterpret_cast<const v4i*>(lds + ((((c * STEPS + s) * 4 + g) * M + j) << 4));
                    acc[s] = mfma(av, b, acc[s]);
                }
            } else {
#pragma unroll
                for (int s = 0; s < STEPS; ++s) {
                    v4i av = v4i{0, 0, 0, 0};
                    if (j < M)
                        av = *reinterpret_cast<const v4i*>(lds + ((((c * STEPS + s) * 4 + g) * M + j) << 4));
                    v4i b;
                    if constexpr (FMT == XT_INT8) {
                        b = wv[t][s];
                    } else if constexpr (FMT == XT_INT4) {
#pragma unroll
                        for (int d = 0; d < 4; ++d)  // tiles hold the codes q + 8
                            b[d] = (int)(((unsigned)wv[t][s >> 1][d] >> (4 * (s & 1))) & 0x0f0f0f0fu);
                    } else {
                        b = decode4(wv[t][0][s]);
                    }
                    acc[s] = mfma(av, b, acc[s]);
                }
            }
        }
    }
#pragma unroll
    for (int s = 1; s < STEPS; ++s) acc[0] += acc[s];

    red[wave][lane] = acc[0];
    __syncthreads();
    if (wave != 0) return;
    v4i sum = v4i{0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < WAVES; ++w) sum += red[w][lane];
    if (o >= N) return;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = 4 * g + r;
        if (i >= M) continue;
        const int d = sum[r] - OFF * rsum[i];
        // layers.rs:294 — (dot as f32 * inv_scale) * w_scale, two roundings.
        y[(size_t)i * N + o] = __fmul_rn(__fmul_rn((float)d, invr[r]), wscale);
        if (accout) accout[(size_t)i * N + o] = d;
    }
}

// LDS budget for staged activations and the chunk bound per wave.
constexpr int kGemvLds = 96 * 1024;

// chunks per wave each compiled GEMV width can hold
int gemv_ncw(int waves) { return waves == 16 ? 4 : waves == 8 ? 8 : 16; }

bool gemv_fits(int fmt, int M, int nch, int waves, int ncw) {
    const int ch = fmt == XT_PACK5 ? 320 : 256;
    return M >= 1 && M <= 16 && (size_t)M * nch * ch <= (size_t)kGemvLds &&
           (nch + waves - 1) / waves <= ncw;
}

// ---------------------------------------------------------------------------
// Decode GEMV for ternary formats without staging (M <= 16, q given)
// ---------------------------------------------------------------------------
//
// Workgroup x owns the 16 output rows of row group x (of the projection x
// falls in) over all of K; wave w takes chunks w, w + WAVES, ...  Every lane
// loads its weight slot and its four (Pack5: five) 16-byte activation pieces
// straight from memory -- no LDS stage, no barrier before the MFMAs -- and all
// loads are unconditional (clamped indices, zero-selected afterwards), so
// they issue back to back.  Codes are decoded to signed weights with one
// v_perm_b32 (code 0 -> -1, 1 -> 0, 2 -> +1, 3 -> 0), so no activation row
// sum is needed.  Waves are summed through LDS once at the end.

// FUSED: the kernel quantises the one f32 row a.x itself (quantization.rs:95-195,
// as quantize_kernel): each lane reads its pieces as f32, the row's absmax
// goes through the waves' shuffles and LDS (one barrier), then each lane
// quantises its own pieces.  No separate quantiser launch.
// AM > 0 (M <= AM, q given): the wave's activation bytes (rows < M of its
// chunks, 256 / 320 bytes each) are loaded once, one distinct 16-byte piece
// per lane, passed through a wave-private LDS slice and read back as MFMA
// fragments, instead of every lane loading its four / five pieces from
// memory (16 token lanes per fragment, most of them duplicates for small M).
template <int FMT, int WAVES, int NCW, bool FUSED, int RG, int AM = 0>
__global__ __launch_bounds__(WAVES * 64) void gemv2_kernel(const MMArgs a) {
    constexpr int STEPS = (FMT == XT_PACK5) ? 5 : 4;
    constexpr int CH = STEPS * 64;
    // 1 KiB tiles per chunk: Int8 one per k-step, Int4 one per two k-steps
    constexpr int TPC = (FMT == XT_INT8) ? 4 : (FMT == XT_INT4 ? 2 : 1);
    constexpr int APR = NCW * CH / 16;                   // pieces per row and wave
    constexpr int APS = APR + 1;                         // row stride in the slice: one
                                                         // piece of padding, so the rows
                                                         // of a fragment read hit distinct banks
    constexpr int APW = AM > 0 ? AM * APR : 1;           // pieces per wave
    constexpr int ALL = (APW + 63) / 64;                 // of them per lane
    __shared__ v4i red[WAVES][RG][64];
    __shared__ v4i aslice[WAVES][AM == 16 ? 16 * 17 : (AM > 0 ? AM * APS : 1)];
    __shared__ unsigned tmax[WAVES][16];
    __shared__ __align__(16) unsigned qrow[FUSED ? WAVES : 1][FUSED ? NCW : 1][FUSED ? CH / 4 : 4];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int g = lane >> 4;
    const int j = lane & 15;
    const int bx = blockIdx.x;
    const int M = a.M;
    const int nch = a.nch;
    const int ldq = a.ldq;
    const int8_t* q = a.q;
    const float* inv = a.inv;
    const ProjBounds pb = proj_bounds();
    __builtin_amdgcn_sched_barrier(0);  // one round of argument loads
    const ProjView pv = select_proj(pb, bx);
    const int N = pv.N;
    const int NG = (N + 15) >> 4;
    const int G0 = (bx - pv.tile0) * RG;  // first row group of the workgroup

    // epilogue operands (wave w < RG finishes row group G0 + w: tokens
    // 4g + r, output row o)
    const int o = (G0 + min(wave, RG - 1)) * 16 + j;
    const float wscale = pv.ws[min(o, N - 1)];
    float invr[4];
    if constexpr (!FUSED) {
#pragma unroll
        for (int r = 0; r < 4; ++r) invr[r] = inv[min(4 * g + r, M - 1)];
    }

    const uint8_t* wsrc[RG];
#pragma unroll
    for (int r = 0; r < RG; ++r)
        wsrc[r] = pv.tiles + ((size_t)min(G0 + r, NG - 1) * nch * TPC * 64 + lane) * 16;
    v4i wv[NCW][RG][TPC];
    v4i av[NCW][STEPS];
    if constexpr (AM == 16) {
        // 9-16 rows of 2-bit tiles: each activation load covers 4 token rows
        // x 256 bytes of one chunk (one instruction spanning 16 rows at the
        // row stride stalls the address path on translation); chunk by
        // chunk the 16 rows go through the wave's LDS slice (rows padded by
        // one piece) and come back as MFMA fragments.
        static_assert(!FUSED && FMT != XT_PACK5, "AM 16: quantised rows, 256-column chunks");
#pragma unroll
        for (int t = 0; t < NCW; ++t) {
            const int c = min(wave + t * WAVES, nch - 1);
#pragma unroll
            for (int u = 0; u < 4; ++u)  // (rows >= M clamped, zeroed at the MFMA)
                av[t][u] = ld_cached(q + (size_t)min(4 * u + (lane >> 4), M - 1) * ldq + (size_t)c * CH +
                                     (lane & 15) * 16);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NCW; ++t) {
            const int c = min(wave + t * WAVES, nch - 1);
#pragma unroll
            for (int r = 0; r < RG; ++r)
#pragma unroll
                for (int u = 0; u < TPC; ++u)
                    wv[t][r][u] = ld_stream(wsrc[r] + ((size_t)c * TPC + u) * kTileBytes);
        }
        __builtin_amdgcn_sched_barrier(0);
        // (a wave's LDS accesses complete in order: each chunk's reads see
        // its stores, and precede the next chunk's stores)
#pragma unroll
        for (int t = 0; t < NCW; ++t) {
#pragma unroll
            for (int u = 0; u < 4; ++u) aslice[wave][(4 * u + (lane >> 4)) * 17 + (lane & 15)] = av[t][u];
            __asm__ volatile("" ::: "memory");
#pragma unroll
            for (int st = 0; st < 4; ++st) av[t][st] = aslice[wave][j * 17 + 4 * st + g];
            __asm__ volatile("" ::: "memory");
        }
    } else if constexpr (AM > 0) {
        static_assert(!FUSED, "AM takes quantised rows");
        const int npc = M * APR;  // pieces of rows < M
        v4i ap[ALL];
#pragma unroll
        for (int u = 0; u < ALL; ++u) {
            const int p = min(lane + 64 * u, npc - 1);
            const int m = p / APR, pr = p - m * APR;
            const int c = min(wave + (pr / (CH / 16)) * WAVES, nch - 1);
            ap[u] = ld_cached(q + (size_t)m * ldq + (size_t)c * CH + (pr % (CH / 16)) * 16);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NCW; ++t) {
            const int c = min(wave + t * WAVES, nch - 1);
#pragma unroll
            for (int r = 0; r < RG; ++r)
#pragma unroll
                for (int u = 0; u < TPC; ++u)
                    wv[t][r][u] = ld_stream(wsrc[r] + ((size_t)c * TPC + u) * kTileBytes);
        }
        __builtin_amdgcn_sched_barrier(0);
        // (a wave's LDS accesses complete in order: the reads below see
        // these stores without a barrier)
#pragma unroll
        for (int u = 0; u < ALL; ++u)
            if (lane + 64 * u < npc) aslice[wave][lane + 64 * u + (lane + 64 * u) / APR] = ap[u];
        __asm__ volatile("" ::: "memory");
        const int jr = min(j, M - 1) * APS;
#pragma unroll
        for (int t = 0; t < NCW; ++t)
#pragma unroll
            for (int s = 0; s < STEPS; ++s) av[t][s] = aslice[wave][jr + t * (CH / 16) + 4 * s + g];
    } else if constexpr (!FUSED) {
        const int8_t* arow = q + (size_t)min(j, M - 1) * ldq + 16 * g;
#pragma unroll
        for (int t = 0; t < NCW; ++t) {
            const int c = min(wave + t * WAVES, nch - 1);
#pragma unroll
            for (int r = 0; r < RG; ++r)
#pragma unroll
                for (int u = 0; u < TPC; ++u)
                    wv[t][r][u] = ld_stream(wsrc[r] + ((size_t)c * TPC + u) * kTileBytes);
#pragma unroll
            for (int s = 0; s < STEPS; ++s) av[t][s] = ld_cached(arow + (size_t)c * CH + s * 64);
        }
    } else {
        const int K = a.K;
        const int n4 = K >> 2;
        // One row: lane l of wave w loads float4 piece l of each chunk the
        // wave multiplies (chunks w + t WAVES), and for Pack5's 80-piece
        // chunks also piece 64 + l (l < 16), so every lane finds its A
        // fragment in the packed bytes of four lanes of its own wave
        // (its LDS row, no stage); the row maximum comes from per-wave
        // maxima (no atomics, so no clearing barrier).  One barrier in all.
        constexpr int PPC = CH / 4;  // float4 pieces per chunk: 64 or 80
        float4 x0[NCW], x1[NCW];
#pragma unroll
        for (int t = 0; t < NCW; ++t) {
            const int f = (wave + t * WAVES) * PPC + lane;
            x0[t] = x1[t] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (f < n4) x0[t] = *reinterpret_cast<const float4*>(a.x + 4 * f);
            if constexpr (PPC > 64)
                if (lane < PPC - 64 && f + 64 < n4) x1[t] = *reinterpret_cast<const float4*>(a.x + 4 * (f + 64));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NCW; ++t) {
            const int c = min(wave + t * WAVES, nch - 1);
#pragma unroll
            for (int r = 0; r < RG; ++r)
#pragma unroll
                for (int u = 0; u < TPC; ++u)
                    wv[t][r][u] = ld_stream(wsrc[r] + ((size_t)c * TPC + u) * kTileBytes);
        }
        __builtin_amdgcn_sched_barrier(0);
        // (non-negative floats order as their bit patterns; NaN is ignored)
        auto amax = [](float4 v) { return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))); };
        float mx = 0.0f;
#pragma unroll
        for (int t = 0; t < NCW; ++t) mx = fmaxf(mx, fmaxf(amax(x0[t]), amax(x1[t])));
        const int wm = wave_reduce_bits(__float_as_int(mx), [](int p, int q) {
            return __float_as_int(fmaxf(__int_as_float(p), __int_as_float(q)));
        });
        if (lane == 0) tmax[wave][0] = (unsigned)wm;
        __syncthreads();
        unsigned mb = 0u;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) mb = max(mb, tmax[w][0]);
        const float rmx = __uint_as_float(mb);
        const float scale = (rmx > 0.0f) ? __fdiv_rn(127.0f, rmx) : 1.0f;
        const float iv = (rmx > 0.0f) ? __fdiv_rn(rmx, 127.0f) : 1.0f;
#pragma unroll
        for (int r = 0; r < 4; ++r) invr[r] = iv;
        const int kmain = (K / 16) * 16;
        unsigned w4[NCW], w5[NCW];
        auto pack = [&](auto mode_c) {
            auto q4 = [&](float4 v, int f) {
                const int col = 4 * f;
                const float e4[4] = {v.x, v.y, v.z, v.w};
                unsigned r = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    r |= (unsigned)(quant_one(e4[e], scale, decltype(mode_c)::value, col + e < kmain) & 255)
                         << (8 * e);
                return f < n4 ? r : 0u;  // columns past K: zero activations
            };
#pragma unroll
            for (int t = 0; t < NCW; ++t) {
                const int f = (wave + t * WAVES) * PPC + lane;
                w4[t] = q4(x0[t], f);
                w5[t] = PPC > 64 ? q4(x1[t], f + 64) : 0u;
            }
        };
        if (a.mode == XT_QUANT_AVX512) pack(std::integral_constant<int, XT_QUANT_AVX512>{});
        else pack(std::integral_constant<int, XT_QUANT_SCALAR>{});
        // The chunk's packed bytes through the wave's LDS row: lane (g, j)
        // of step s reads pieces 16 s + 4 g .. + 3, the same 16 bytes for
        // every j (one write and four broadcast reads per chunk against
        // 16 ds_bpermute: 2560 -> 640 4.32 -> 3.86 us, 6912 -> 2560 5.81 ->
        // 5.64).  A wave's LDS accesses complete in order: no barrier.
#pragma unroll
        for (int t = 0; t < NCW; ++t) {
            qrow[wave][t][lane] = w4[t];
            if constexpr (PPC > 64)
                if (lane < PPC - 64) qrow[wave][t][64 + lane] = w5[t];
        }
        __asm__ volatile("" ::: "memory");
#pragma unroll
        for (int t = 0; t < NCW; ++t)
#pragma unroll
            for (int st = 0; st < STEPS; ++st)
                av[t][st] = *reinterpret_cast<const v4i*>(&qrow[wave][t][16 * st + 4 * g]);
    }
    v4i acc[RG][STEPS];
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
        for (int s = 0; s < STEPS; ++s) acc[r][s] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int t = 0; t < NCW; ++t) {
        // (A rows >= M only reach sums that are not stored, and the fused
        // quantiser's chunks past the row are zeros: no select there.  Skipping
        // such chunks, or leaving the select to them alone, was slower at
        // M = 16, 14336 -> 4096: 8.0 -> 8.6 us)
        const bool live = FUSED || wave + t * WAVES < nch;
#pragma unroll
        for (int r = 0; r < RG; ++r) {
            if constexpr (FMT == XT_PACK5) {
                int E[4], O[4];
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    E[d] = wv[t][r][0][d] & 0x00ff00ff;
                    O[d] = ((unsigned)wv[t][r][0][d] >> 8) & 0x00ff00ff;
                }
#pragma unroll
                for (int s = 0; s < STEPS; ++s) {
                    v4i b;
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        const int pE = E[d] * 3, pO = O[d] * 3;
                        b[d] = signed_codes((int)__builtin_amdgcn_perm((unsigned)pO, (unsigned)pE, 0x07030501u));
                        E[d] = pE & 0x00ff00ff;
                        O[d] = pO & 0x00ff00ff;
                    }
                    const v4i x = FUSED || (live && j < M) ? av[t][s] : v4i{0, 0, 0, 0};
                    acc[r][s] = mfma(x, b, acc[r][s]);
                }
            } else {
#pragma unroll
                for (int s = 0; s < STEPS; ++s) {
                    v4i b;
                    if constexpr (FMT == XT_INT8) {
                        b = wv[t][r][s];
                    } else if constexpr (FMT == XT_INT4) {
                        // code c = q + 8 -> (c ^ 8) in the high nibble is the
                        // signed byte 16 q; the sum is divided by 16 at the end
#pragma unroll
                        for (int d = 0; d < 4; ++d) {
                            const unsigned w = (unsigned)wv[t][r][s >> 1][d] ^ 0x88888888u;
                            b[d] = (int)(((s & 1) ? w : (w << 4)) & 0xf0f0f0f0u);
                        }
                    } else {
                        b = decode4(wv[t][r][0][s]);
#pragma unroll
                        for (int d = 0; d < 4; ++d) b[d] = signed_codes(b[d]);
                    }
                    const v4i x = FUSED || (live && j < M) ? av[t][s] : v4i{0, 0, 0, 0};
                    acc[r][s] = mfma(x, b, acc[r][s]);
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < RG; ++r) {
#pragma unroll
        for (int s = 1; s < STEPS; ++s) acc[r][0] += acc[r][s];
        red[wave][r][lane] = acc[r][0];
    }
    __syncthreads();
    if (wave >= RG || o >= N) return;
    v4i sum = red[0][wave][lane];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sum += red[w][wave][lane];
    if constexpr (FMT == XT_INT4) {
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[r] >>= 4;  // exact: every term is a multiple of 16
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = 4 * g + r;
        if (i >= M) continue;
        // layers.rs:294 — (dot as f32 * inv_scale) * w_scale, two roundings.
        pv.y[(size_t)i * N + o] = __fmul_rn(__fmul_rn((float)sum[r], invr[r]), wscale);
        if (pv.acc) pv.acc[(size_t)i * N + o] = sum[r];
    }
}

// Row groups per workgroup of the staging-free GEMV: the most (4, 2, 1)
// that leave at least 200 workgroups and at most 80 KiB of weights per
// workgroup.  Measured (MI355X, rotating weights, µs at M = 1 / 16 for 1, 2,
// 4 groups): C0 2560 -> 6912 3.7 / 3.5 / 4.1 at M = 1; 4096 -> 14336 7.5 /
// 5.9 / 5.3 and 11.8 / 7.9 / 6.4; 2560 -> 32768 at M = 16 14.3 / 11.1 / 7.8;
// Int4 head 128256 rows 33.3 / 29.7 / 27.9; Int8 head 48.9 / 49.9 / 52.1 at
// M = 1 and 72.6 / 61.9 / 61.1 at M = 16.  Pack5 never takes two (3200 ->
// 8640: 5.3 / 6.1 / 6.1; 3200 -> 32000: 11.0 / 12.1 / 9.3).
static int gemv2_rg_for(int fmt, int nch, int ngroups) {
    const int tpc = fmt == XT_INT8 ? 4 : (fmt == XT_INT4 ? 2 : 1);
    for (int rg : {4, 2})
        if (ngroups / rg >= 200 && rg * nch * tpc * kTileBytes <= 80 * 1024 &&
            !(fmt == XT_PACK5 && rg == 2))
            return rg;
    return 1;
}

// Chunks of the longest f32 row that the GEMV quantises itself; longer rows
// take the quantiser launch.  Below the line the fused form saves that launch
// (launch to launch, us, fused / with the launch, to 640 outputs: Pack4 4096
// 3.4 / 5.3, 9216 5.7 / 7.4; Pack5 8960 6.9 / 7.8).  The line is no optimum:
// it lies where the LDS stage of an earlier form that took several rows ended,
// and the one-row form would gain beyond it as well (Pack4 9472 5.9 / 7.5,
// 16384 7.3 / 8.9; Pack5 9280 7.0 / 7.8).
constexpr int fused_chunks(int fmt) { return fmt == XT_PACK5 ? 28 : 36; }
bool gemv2_fuses(int fmt, int nch) { return nch <= fused_chunks(fmt); }

// Quantised rows given: the activation pieces through a wave-private LDS
// slice when the wave multiplies two or more chunks and the slice of M rows
// fits (measured: 14336 -> 4096 at M = 1 / 4 6.42 -> 5.24-5.39 / 6.93 ->
// 6.04 us; Pack5 3200 -> 8640 at M = 1 / 8 4.80 -> 4.48-4.54 / 5.99 ->
// 5.23; with one chunk per wave it did not help: 4096 -> 14336 at M = 1
// 5.33 -> 5.55).
template <int FMT, int W, int NCW, int RG, int AM>
static constexpr bool gemv2_am_fits() {
    return (size_t)W * AM * (NCW * (FMT == XT_PACK5 ? 320 : 256) + 16) + (size_t)W * RG * 1024 <= 120 * 1024;
}
template <int FMT, int W, int NCW, int RG>
static hipError_t launch_gemv2_am(const MMArgs& a, int ntiles, hipStream_t s) {
    const dim3 g(ntiles), b(W * 64);
    if constexpr (NCW >= 2) {
        if (a.M == 1) {
            hipLaunchKernelGGL((gemv2_kernel<FMT, W, NCW, false, RG, 1>), g, b, 0, s, a);
            return hipGetLastError();
        }
        if constexpr (gemv2_am_fits<FMT, W, NCW, RG, 4>()) {
            if (a.M <= 4) {
                hipLaunchKernelGGL((gemv2_kernel<FMT, W, NCW, false, RG, 4>), g, b, 0, s, a);
                return hipGetLastError();
            }
        }
        if constexpr (gemv2_am_fits<FMT, W, NCW, RG, 8>()) {
            if (a.M <= 8) {
                hipLaunchKernelGGL((gemv2_kernel<FMT, W, NCW, false, RG, 8>), g, b, 0, s, a);
                return hipGetLastError();
            }
        }
    }
    // 5-16 rows of 2-bit tiles the slices above do not take: 4-row loads,
    // staged chunk by chunk (measured: TA address stalls 68 % -> see the
    // profile of this kernel)
    if constexpr (FMT == XT_PACK4 && (size_t)W * (16 * 17 * 16 + RG * 1024) <= 150 * 1024) {
        if (a.M > 4 && a.M <= 16) {
            hipLaunchKernelGGL((gemv2_kernel<FMT, W, NCW, false, RG, 16>), g, b, 0, s, a);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((gemv2_kernel<FMT, W, NCW, false, RG>), g, b, 0, s, a);
    return hipGetLastError();
}

// Int8 rows given: 5-16 rows take the 4-row activation loads staged through
// the LDS slice, as the ternary tiles do (measured on the 128256-row head at
// M = 16: Int8 63.2 -> 60.2 us; Int4 36.4 -> 38.1, so Int4 keeps the direct
// loads).
template <int FMT, int W, int NCW, int RG>
static hipError_t launch_gemv2_int(const MMArgs& a, int ntiles, hipStream_t s) {
    const dim3 g(ntiles), b(W * 64);
    if constexpr (FMT == XT_INT8 && (size_t)W * (16 * 17 * 16 + RG * 1024) <= 150 * 1024) {
        if (a.M > 4 && a.M <= 16) {
            hipLaunchKernelGGL((gemv2_kernel<FMT, W, NCW, false, RG, 16>), g, b, 0, s, a);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((gemv2_kernel<FMT, W, NCW, false, RG>), g, b, 0, s, a);
    return hipGetLastError();
}

// One f32 row quantised in the kernel: compiled for the waves and chunks per
// wave that rows of up to fused_chunks(FMT) reach (14 x 2 for Pack5, 14 x 3
// for Pack4).
template <int FMT, int W, int NCW, int RG>
static hipError_t launch_gemv2_fused(const MMArgs& a, int ntiles, hipStream_t s) {
    if constexpr (W * NCW <= (fused_chunks(FMT) + 13) / 14 * 14) {
        hipLaunchKernelGGL((gemv2_kernel<FMT, W, NCW, true, RG>), dim3(ntiles), dim3(W * 64), 0, s, a);
        return hipGetLastError();
    }
    return hipErrorInvalidValue;
}

// The staging-free GEMV applies to ternary tiles (given or fused-quantised rows).
template <int RG>
static hipError_t launch_gemv2_rg(int fmt, const MMArgs& a, int ntiles, hipStream_t s) {
    const int nch = a.nch;
    if (a.x && (a.M != 1 || !gemv2_fuses(fmt, nch))) return hipErrorInvalidValue;
#define XT_GV2(W_, NCW_)                                                                         \
    if (nch <= W_ * NCW_) {                                                                      \
        if (a.x) {                                                                               \
            if (fmt == XT_PACK5)                                                                 \
                return launch_gemv2_fused<XT_PACK5, W_, NCW_, RG>(a, ntiles, s);                 \
            return launch_gemv2_fused<XT_PACK4, W_, NCW_, RG>(a, ntiles, s);                     \
        } else if (fmt == XT_PACK5) {                                                            \
            return launch_gemv2_am<XT_PACK5, W_, NCW_, RG>(a, ntiles, s);                      \
        } else if (fmt == XT_INT8) {                                                             \
            if constexpr (NCW_ <= 2)                                                             \
                return launch_gemv2_int<XT_INT8, W_, NCW_, RG>(a, ntiles, s);                        \
            else                                                                                 \
                return hipErrorInvalidValue;                                                     \
        } else if (fmt == XT_INT4) {                                                             \
            if constexpr (NCW_ <= 2)                                                             \
                return launch_gemv2_int<XT_INT4, W_, NCW_, RG>(a, ntiles, s);                        \
            else                                                                                 \
                return hipErrorInvalidValue;                                                     \
        } else {                                                                                 \
            return launch_gemv2_am<XT_PACK4, W_, NCW_, RG>(a, ntiles, s);                      \
        }                                                                                        \
    }
    // Pack5 at 5..10 chunks: five waves of two chunks (measured, 3200 ->
    // 8640: 4.8 vs 5.3 us at M = 1, 6.0 vs 6.2 at M = 8; Pack4 is fastest
    // with one chunk per wave)
    if (fmt == XT_PACK5 && !a.x && nch > 4 && nch <= 10) {
        return launch_gemv2_am<XT_PACK5, 5, 2, RG>(a, ntiles, s);
        return hipGetLastError();
    }
    // Above 16 chunks, 14 waves where they cover K with the same chunks per
    // wave (27 or 28 chunks, 42, 56): fewer idle waves (measured at M = 1 /
    // 8: 6912 -> 2560 4.3 -> 4.1 / 5.3 -> 5.0 us; 14336 -> 4096 6.7 -> 6.3 /
    // 8.3 -> 7.7; Pack5 8640 -> 3200 5.1 -> 5.0 / 5.6 -> 5.5)
    XT_GV2(4, 1) XT_GV2(8, 1) XT_GV2(10, 1) XT_GV2(16, 1) XT_GV2(14, 2) XT_GV2(16, 2)
    XT_GV2(14, 3) XT_GV2(16, 3) XT_GV2(14, 4) XT_GV2(16, 4)
#undef XT_GV2
    return hipErrorInvalidValue;
}

static hipError_t launch_gemv2(int fmt, const MMArgs& a, int ntiles, hipStream_t s) {
    if (a.rg == 4) return launch_gemv2_rg<4>(fmt, a, ntiles, s);
    return a.rg == 2 ? launch_gemv2_rg<2>(fmt, a, ntiles, s) : launch_gemv2_rg<1>(fmt, a, ntiles, s);
}

static bool use_gemv2(int fmt, int nch) {
    if (fmt == XT_INT8 || fmt == XT_INT4) return nch <= 32;  // weight registers: 4 / 2 tiles a chunk
    return (fmt == XT_PACK4 || fmt == XT_PACK5 || fmt == XT_XORSPARSE) && nch <= 64;
}
bool gemv2_takes(int fmt, int nch) { return use_gemv2(fmt, nch); }
int gemv_row_groups(int fmt, int nch, int ngroups) {
    return use_gemv2(fmt, nch) ? gemv2_rg_for(fmt, nch, ngroups) : 1;
}

hipError_t launch_gemv(int fmt, const MMArgs& a, int ntiles, int waves, hipStream_t s) {
    // (Int8 / Int4 rows quantised in the kernel stay on the staged GEMV)
    if (use_gemv2(fmt, a.nch) && !(a.x && is_int_format(fmt)))
        return launch_gemv2(fmt == XT_XORSPARSE ? XT_PACK4 : fmt, a, ntiles, s);
    const int ch = fmt == XT_PACK5 ? 320 : 256;
    const size_t lds = (size_t)a.M * a.nch * ch;
#define XT_GEMV(W_, NCW_)                                                                        \
    if (waves == W_) {                                                                           \
        if (fmt == XT_PACK5)                                                                     \
            hipLaunchKernelGGL((gemv_kernel<XT_PACK5, W_, NCW_>), dim3(ntiles), dim3(W_ * 64), lds, s, a); \
        else if (fmt == XT_INT8)                                                                 \
            hipLaunchKernelGGL((gemv_kernel<XT_INT8, W_, NCW_>), dim3(ntiles), dim3(W_ * 64), lds, s, a); \
        else if (fmt == XT_INT4)                                                                 \
            hipLaunchKernelGGL((gemv_kernel<XT_INT4, W_, NCW_>), dim3(ntiles), dim3(W_ * 64), lds, s, a); \
        else                                                                                     \
            hipLaunchKernelGGL((gemv_kernel<XT_PACK4, W_, NCW_>), dim3(ntiles), dim3(W_ * 64), lds, s, a); \
        return hipGetLastError();                                                                \
    }
    XT_GEMV(4, 16)
    XT_GEMV(8, 8)
    XT_GEMV(2, 16)
    XT_GEMV(16, 4)
#undef XT_GEMV
    return hipErrorInvalidValue;
}

// Compiled tile shapes, selectable by MMConfig; (1, 1, 4, 4), (1, 4, 4, 2) and
// (2, 8, 4, 2) run only when forced, and carry the tests of split K.
#define XT_MM_SHAPES(X)  \
    X(1, 1, 4, 4)        \
    X(1, 1, 8, 2)        \
    X(1, 2, 4, 4)        \
    X(1, 4, 4, 2)        \
    X(1, 4, 8, 2)        \
    X(1, 5, 8, 2)        \
    X(1, 8, 8, 2)        \
    X(1, 5, 16, 1)       \
    X(2, 8, 4, 2)

namespace {
bool shape_known(const MMConfig& c, bool own) {
#define XT_KNOWN(MB_, NB_, W_, PF_) \
    if (c.mb == MB_ && c.nb == NB_ && c.waves == W_ && c.pf == PF_) return !own || MB_ == 1;
    XT_MM_SHAPES(XT_KNOWN)
#undef XT_KNOWN
    return false;
}

// XTERN_CONFIG="mb,nb,waves,pf,splitk" forces one tile shape (for tuning; the
// only way to splitk > 1 slices of K over workgroups), "gw,mw,nw,waves" one
// shape of the many-row GEMM, "gemv,W" the decode GEMV.
bool env_config(MMConfig* c) {
    const char* e = getenv("XTERN_CONFIG");
    MMConfig f;
    int mw = 0, nw = 0, w = 0;
    if (e && sscanf(e, "gw,%d,%d,%d", &mw, &nw, &w) == 3) {
        f = MMConfig{2 * mw, 2 * nw * w, w, 1, 1};
        f.kind = 4;
        *c = f;
        return true;
    }
    if (e && sscanf(e, "gemv,%d", &f.waves) == 1) {
        f = MMConfig{1, 1, f.waves, 1, 1};
        f.kind = 2;
        *c = f;
        return true;
    }
    if (e && sscanf(e, "%d,%d,%d,%d,%d", &f.mb, &f.nb, &f.waves, &f.pf, &f.splitk) == 5 &&
        f.splitk >= 1) {
        *c = f;
        return true;
    }
    return false;
}
}  // namespace

// Waves per workgroup of the Int8 / Int4 GEMV for row blocks of mb tokens.
int int_gemv_waves(int fmt, int mb, int nch) {
    MMConfig c;
    if (env_config(&c) && c.kind == 2 && gemv_fits(fmt, mb, nch, c.waves, gemv_ncw(c.waves)))
        return c.waves;
    // Measured on the 128256 x 2560 LM head: Int4 streams fastest with 8
    // waves (46.5 vs 58 us at M = 1), Int8 with 16.
    return (fmt == XT_INT4 && gemv_fits(fmt, mb, nch, 8, gemv_ncw(8))) ? 8 : 16;
}

namespace {
// Shapes of a product with more than 16 rows, and what one of them costs in
// microseconds: `start` once; per chunk of K (K in rounds of `unit` chunks)
// `first` for a workgroup that has its CU to itself, `rest` for each further
// one of the busiest CU, and `gap` once per further one (its start and
// epilogue, as far as they are not hidden).  `spread`: mm_kernel's workgroup t
// runs on XCD t % 8, so a column of weights that more than one XCD multiplies
// is read into the L2 of each; per chunk, with all 8 of them and every CU
// taken.  `acts`: most KiB of activations (0: any).
// Pack4: fitted to launch-to-launch times on MI355X of all eight shapes at
// 2047 sizes (M = 17 .. 4096, K = 256 .. 14336, N = 100 .. 17280, weights
// streamed from memory): the shape chosen is 0.8 % slower than the fastest on
// average and within 3 % of it at nine sizes of ten.
struct GemmShape {
    int mb, nb, waves, pf, kind;
    float start, first, spread, rest, gap;
    int unit, acts;
};
// 16-token shapes (mm_kernel) win while every CU gets at most one of them, 32
// output rows before 64 and more (the smallest start; us, 16 x 32 / 16 x 64 /
// 32 x 128: 4096 -> 2560 at M = 17 5.3 / 5.8 / 8.3, 4096 -> 640 at M = 128
// 5.0 / 6.2 / 7.9), except that its many columns read large activations again
// and again (14336 -> 256 at M = 512: 15.4 / 13.3); 16 x 128 where its columns
// divide over the XCDs (/ 32 x 128: 5120 -> 4096 at M = 128 8.6 / 10.0, but
// 4096 -> 3200 10.9 / 8.2); then ever larger tiles of gemmw_kernel.  Examples,
// us (16 x 64 / 16 x 128 / 32 x 128 / 64 x 128 / 64 x 256 / 128 x 256): 2560
// -> 6912 at M = 32 6.2 / 7.4 / 6.7 / 9.4 / 13 / 20, at M = 512 - / - / 16.5 /
// 14.2 / 14.0 / 20.4, at M = 2048 - / - / 47 / 41 / 39 / 38; 6912 -> 2560 at
// M = 64 7.9 / 10.7 / 11.9 / 13.9 / 22 / 42, at M = 512 - / - / 18.7 / 15.9 /
// 24 / 39.
const GemmShape kShapes4[] = {
    {1, 2, 4, 4, 0, 2.54f, 0.150f, 0.099f, 0.170f, 1.00f, 1, 1750},
    {1, 4, 8, 2, 0, 2.80f, 0.145f, 0.128f, 0.160f, 1.20f, 1, 0},
    {1, 5, 8, 2, 0, 3.18f, 0.143f, 0.157f, 0.190f, 1.20f, 1, 0},
    {1, 8, 8, 2, 0, 3.31f, 0.260f, 0.123f, 0.245f, 1.20f, 1, 0},
    {2, 8, 4, 1, 4, 2.40f, 0.338f, 0.0f, 0.294f, 0.45f, 1, 0},
    {4, 8, 4, 1, 4, 3.09f, 0.396f, 0.0f, 0.437f, 0.95f, 1, 0},
    {4, 16, 4, 1, 4, 3.82f, 0.850f, 0.0f, 0.826f, 0.82f, 1, 0},
    {8, 16, 4, 1, 4, 4.65f, 1.673f, 0.0f, 1.316f, 1.38f, 1, 0},
};
// Pack5 (the base-3 decode is 24 vector instructions per 16 weights against
// 9, so shapes that decode a weight once for 128 tokens pay earlier): 3200 ->
// 8640, 32 x 128 / 64 x 128 / 128 x 128 / 128 x 256 (eight waves): M = 128
// 15.5 / 12.2 / 16.6 / 22.1, M = 512 32 / 27.8 / 33.7 / 25.6, M = 2048 103 /
// 77 / 83 / 75.
const GemmShape kShapes5[] = {
    {1, 2, 4, 4, 0, 0.0f, 0.290f, 0.0f, 0.160f, 0.0f, 1, 0},
    {1, 4, 8, 2, 0, 0.0f, 0.270f, 0.0f, 0.200f, 0.0f, 8, 0},
    {1, 5, 8, 2, 0, 0.0f, 0.310f, 0.0f, 0.220f, 0.0f, 8, 0},
    {1, 5, 16, 1, 0, 0.0f, 0.275f, 0.0f, 0.360f, 0.0f, 16, 0},
    {2, 8, 4, 1, 4, 0.0f, 0.650f, 0.0f, 0.500f, 0.8f, 1, 0},
    {4, 8, 4, 1, 4, 0.0f, 0.800f, 0.0f, 0.620f, 2.2f, 1, 0},
    {8, 8, 4, 1, 4, 0.0f, 1.300f, 0.0f, 1.300f, 3.0f, 1, 0},
    {8, 16, 8, 1, 4, 0.0f, 2.000f, 0.0f, 2.200f, 3.5f, 1, 0},
};

// gemmw_kernel's byte offsets within a matrix and a token block are 32-bit.
bool gemmw_offsets(int ngroups, int nch) {
    return (size_t)ngroups * nch * kTileBytes < ((size_t)1 << 32) && nch < (1 << 16);
}

MMConfig choose_gemm(int fmt, int M, int ngroups, int nch) {
    const bool wide = gemmw_offsets(ngroups, nch);
    MMConfig best;
    double best_cost = -1.0;
    auto take = [&](const GemmShape& g) {
        const long blocks = (M + 16 * g.mb - 1) / (16 * g.mb);
        const long columns = (ngroups + g.nb - 1) / g.nb;
        const long tiles = blocks * columns;
        if (g.acts > 0 && (long)M * nch > g.acts * 4L) return;  // (256 bytes a chunk)
        if (g.kind == 4 && (!wide || tiles > 0x7fffffff)) return;
        // (mm_kernel's row blocks are its grid's y; gemmw_kernel's grid has x only)
        if (g.kind == 0 && wide && blocks > 65535) return;
        const long n = (tiles + 255) / 256;  // workgroups of the busiest CU
        const double nc = (nch + g.unit - 1) / g.unit * g.unit;
        const long period = columns % 8 == 0 ? 1 : columns % 4 == 0 ? 2 : columns % 2 == 0 ? 4 : 8;
        const double others = (double)(std::min(blocks, period) - 1) / 7.0;  // XCDs that read a column again
        const double used = (double)std::min(tiles, 256L) / 256.0;
        const double cost = g.start + nc * (g.first + g.spread * others * used) +
                            (double)(n - 1) * (g.rest * nc + g.gap);
        if (best_cost >= 0.0 && cost >= best_cost) return;
        best_cost = cost;
        best = MMConfig{g.mb, g.nb, g.waves, g.pf, 1, g.kind};
    };
    if (fmt == XT_PACK5)
        for (const GemmShape& g : kShapes5) take(g);
    else
        for (const GemmShape& g : kShapes4) take(g);
    return best;
}
}  // namespace

MMConfig choose_config(int fmt, int M, int ntiles_nb1, int nch, bool have_rowsum) {
    MMConfig c;
    if (env_config(&c)) {
        if (c.kind == 2 && M <= 16 && gemv_fits(fmt, M, nch, c.waves, gemv_ncw(c.waves))) {
            c.nb = gemv_row_groups(fmt, nch, ntiles_nb1);
            return c;
        }
        // (a forced shape of the many-row GEMM is taken or refused: kind -1)
        if (c.kind == 4 && M > 16) {
            if (!gemmw_known(fmt, c.mb / 2, c.waves > 0 ? c.nb / (2 * c.waves) : 0, c.waves) ||
                !gemmw_offsets(ntiles_nb1, nch))
                c.kind = -1;
            return c;
        }
        if (c.kind == 0 && shape_known(c, !have_rowsum)) {
            if (c.splitk > nch) c.splitk = nch;
            return c;
        }
    }
    if (M <= 16) {
        // Measured (MI355X, rotating weights, M = 1..16): the staging-free
        // GEMV wins or ties everywhere, also for many rows (K 2560 -> 8192,
        // M = 4: 3.9 vs 4.7 us on the 32-row, 4-wave K-split kernel;
        // 4096 -> 14336, M = 16: 7.9 vs 8.7).
        if (nch <= 64 || gemv_fits(fmt, M, nch, 16, gemv_ncw(16))) {
            c = MMConfig{1, gemv_row_groups(fmt, nch, ntiles_nb1), 16, 1, 1};
            c.kind = 2;
            return c;
        }
        return MMConfig{1, 1, 8, 2, 1};
    }
    return choose_gemm(fmt, M, ntiles_nb1, nch);
}

hipError_t launch_mm(int fmt, const MMConfig& cfg, const MMArgs& a, int ntiles_total,
                     hipStream_t s) {
    const bool own = (a.rowsum == nullptr);
    const int sk = cfg.splitk;
#define XT_LAUNCH(MB_, NB_, W_, PF_)                                                          \
    if (cfg.mb == MB_ && cfg.nb == NB_ && cfg.waves == W_ && cfg.pf == PF_) {                \
        if constexpr (MB_ == 1) {                                                              \
            if (own)                                                                           \
                return fmt == XT_PACK5                                                         \
                           ? launch_t<XT_PACK5, MB_, NB_, W_, PF_, true>(a, ntiles_total, sk, s) \
                           : launch_t<XT_PACK4, MB_, NB_, W_, PF_, true>(a, ntiles_total, sk, s); \
        }                                                                                      \
        if (own) return hipErrorInvalidValue;                                                  \
        return fmt == XT_PACK5 ? launch_t<XT_PACK5, MB_, NB_, W_, PF_, false>(a, ntiles_total, sk, s) \
                               : launch_t<XT_PACK4, MB_, NB_, W_, PF_, false>(a, ntiles_total, sk, s); \
    }
    XT_MM_SHAPES(XT_LAUNCH)
#undef XT_LAUNCH
    return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------
// HF prepacked weights -> device tiles (src/loader/mod.rs:301-394)
// ---------------------------------------------------------------------------

// The checkpoint stores U8 bytes [R][K], R = N/f, whose digit j (Pack4: bits
// 2j..2j+1, Pack5: base-3 digit j) of byte [p][i] is the weight of output row
// j*R + p at input column i.  One thread builds the 16 bytes of one lane of
// one tile (geometry in xtern_internal.h), reading the digits it needs
// straight from the striped bytes, so the loader's host-side unpack /
// transpose / repack is not needed.  Pack4 code 11 reads as weight 0, as
// unpack_1_58bit_4pack does (quantization.rs:36-41); Pack5 digits are the
// repeated %3, /3 of unpack_1_58bit_5pack (:72-91).
template <int FMT>
__global__ void __launch_bounds__(256)
hf_tiles_kernel(const uint8_t* __restrict__ stored, int64_t K, int64_t N, int64_t R, int64_t nch,
                int64_t nlanes, uint8_t* __restrict__ tiles) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= nlanes) return;
    const int lane = (int)(t & 63);
    const int64_t tile = t >> 6;
    const int64_t G = tile / nch, c = tile % nch;
    const int g = lane >> 4, jr = lane & 15;
    const int64_t o = G * 16 + jr;
    const bool row_ok = o < N;
    const int64_t js = row_ok ? o / R : 0, p = row_ok ? o % R : 0;
    const uint8_t* src = stored + p * K;
    uint32_t out[4];
    if constexpr (FMT == XT_PACK5) {
        const unsigned div = js == 0 ? 1u : js == 1 ? 3u : js == 2 ? 9u : js == 3 ? 27u : 81u;
        uint8_t bytes[16];
#pragma unroll
        for (int b = 0; b < 16; ++b) {
            unsigned v = 0;
#pragma unroll
            for (int st = 0; st < 5; ++st) {
                const int64_t k = c * 320 + st * 64 + g * 16 + b;
                const unsigned code = (row_ok && k < K) ? (src[k] / div) % 3u : 1u;
                v = v * 3u + code;
            }
            bytes[b] = (uint8_t)((v * 256u + 242u) / 243u);
        }
#pragma unroll
        for (int w = 0; w < 4; ++w)
            out[w] = (uint32_t)bytes[4 * w] | ((uint32_t)bytes[4 * w + 1] << 8) |
                     ((uint32_t)bytes[4 * w + 2] << 16) | ((uint32_t)bytes[4 * w + 3] << 24);
    } else {
        const int sh = (int)(2 * js);
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            uint32_t d = 0;
#pragma unroll
            for (int b = 0; b < 16; ++b) {
                const int64_t k = c * 256 + st * 64 + g * 16 + b;
                unsigned code = 1u;
                if (row_ok && k < K) {
                    const unsigned f = (src[k] >> sh) & 3u;
                    code = f == 0u ? 0u : (f == 2u ? 2u : 1u);
                }
                d |= code << (8 * (b & 3) + 2 * (b >> 2));
            }
            out[st] = d;
        }
    }
    *reinterpret_cast<uint4*>(tiles + t * 16) = make_uint4(out[0], out[1], out[2], out[3]);
}

hipError_t launch_hf_tiles(int fmt, const uint8_t* stored, int64_t K, int64_t N, uint8_t* tiles,
                           hipStream_t s) {
    const int64_t f = fmt == XT_PACK5 ? 5 : 4;
    const int64_t nch = (K + chunk_cols(fmt) - 1) / chunk_cols(fmt);
    const int64_t nlanes = (N + 15) / 16 * nch * 64;
    const int64_t blocks = (nlanes + 255) / 256;
    if (blocks > 0x7fffffff) return hipErrorInvalidValue;
    if (fmt == XT_PACK5)
        hipLaunchKernelGGL(hf_tiles_kernel<XT_PACK5>, dim3((unsigned)blocks), dim3(256), 0, s,
                           stored, K, N, N / f, nch, nlanes, tiles);
    else
        hipLaunchKernelGGL(hf_tiles_kernel<XT_PACK4>, dim3((unsigned)blocks), dim3(256), 0, s,
                           stored, K, N, N / f, nch, nlanes, tiles);
    return hipGetLastError();
}

}  // namespace xt
