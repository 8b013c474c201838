// FP8 (OCP e4m3) expert-GEMM path for MoE on MI355X: fp8 matrix instructions
// of its own for the experts.
//
// gfx950 fp8 is OCP e4m3fn (NOT MI300X fnuz — CDNA guide §4). Weights are
// quantized per output row (scale = absmax/448); activations per token.
//
// Three kernels:
//   oa_quant_fp8    bf16 [T, K] -> fp8 [T, K] + f32 scales [T]
//   oa_gemv_fp8     skinny M <= 8 decode path: fp8 W stream (HALF the bytes
//                   of bf16 -> ~2x decode speed for expert projections),
//                   bf16 x, in-register HW dequant (v_cvt_pk_f32_fp8)
//   oa_gemm_fp8     MFMA tile GEMM for prefill-sized M:
//                   C[M,N] = (A8 @ B8^T) * a_scale[m] * b_scale[n] on
//                   v_mfma_f32_16x16x32_fp8_fp8, 128x128 LDS-staged tiles
//                   (the CDNA guide ladder's step-2 structure)

#include "common.h"

typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(2))) int i32x2;

__device__ __forceinline__ u32x4 nt_load4f(const uint32_t* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}

#define FP8_MAX 448.0f

// convert 2 packed fp8 (low/high half-word of src selected by WORD) to floats
template <bool WORD>
__device__ __forceinline__ f32x2 fp8x2_to_f32(unsigned int src) {
    return __builtin_amdgcn_cvt_pk_f32_fp8(src, WORD);
}

// pack two floats into 2 fp8 within `old`'s selected half-word
template <bool WORD>
__device__ __forceinline__ unsigned int f32x2_to_fp8(float a, float b,
                                                     unsigned int old) {
    return __builtin_amdgcn_cvt_pk_fp8_f32(a, b, old, WORD);
}

// ---- per-token quantization -------------------------------------------------
// q[t] = x[t] / scale, scale = max |x[t]| / 448, TPR threads per row: a block or a wave. SILU:
// the row is silu(g) * u of the two halves of x [T, 2 K], rounded to bf16 as the plain
// activation kernel's result is. A thread's first 64 columns stay in registers between the
// two passes, the rest are read again. Bound by the launch up to some MB, by memory above; us, a wave
// per row reading twice / here: [700, 14336] 14.9 / 7.4, [3, 28672] 18.0 / 7.5, [700, 4096]
// in a run of products 9 / 5. SILU with it takes 48 us from a layer's 401 at 700 rows
// (two copies, the activation and a second pass over 20 MB).
template <bool SILU, int TPR>
__global__ __launch_bounds__(256) void quant_fp8_kernel(
    const uint4* __restrict__ x,     // [T, K/8] bf16x8 (SILU: [T, 2 K/8])
    uint2* __restrict__ q,           // [T, K/8] fp8x8
    float* __restrict__ scales,      // [T]
    int T, int kv /* K / 8 */) {
    constexpr int NV = 8;
    const int tid = threadIdx.x & (TPR - 1);
    const size_t row = blockIdx.x * (size_t)(256 / TPR) + threadIdx.x / TPR;
    if (TPR < 256 && row >= T) return;
    const uint4* xr = x + row * kv * (SILU ? 2 : 1);
    uint2* qr = q + row * kv;
    auto load = [&](int c) {
        uint4 w = xr[c];
        if (SILU) {
            const uint4 u = xr[kv + c];
#pragma unroll
            for (int j = 0; j < 4; ++j) (&w.x)[j] = silu_mul_bf16x2((&w.x)[j], (&u.x)[j]);
        }
        return w;
    };
    float amax = 1e-8f;
    auto widen = [&](const uint4& w) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            amax = fmaxf(amax, fmaxf(fabsf(bf16_lo((&w.x)[j])), fabsf(bf16_hi((&w.x)[j]))));
    };
    uint4 w[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int c = v * TPR + tid;
        if (c < kv) widen(w[v] = load(c));
    }
    for (int c = NV * TPR + tid; c < kv; c += TPR) widen(load(c));
    amax = wave_reduce_max(amax);
    if (TPR == 256) {
        __shared__ float red[4];
        if ((threadIdx.x & (WAVE - 1)) == 0) red[threadIdx.x / WAVE] = amax;
        __syncthreads();
        amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    }
    const float inv = FP8_MAX / amax;
    if (tid == 0) scales[row] = amax / FP8_MAX;
    auto store = [&](int c, const uint4& w) {
        uint2 o;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t w0 = (&w.x)[h * 2], w1 = (&w.x)[h * 2 + 1];
            (&o.x)[h] = f32x2_to_fp8<true>(
                bf16_lo(w1) * inv, bf16_hi(w1) * inv,
                f32x2_to_fp8<false>(bf16_lo(w0) * inv, bf16_hi(w0) * inv, 0));
        }
        qr[c] = o;
    };
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int c = v * TPR + tid;
        if (c < kv) store(c, w[v]);
    }
    for (int c = NV * TPR + tid; c < kv; c += TPR) store(c, load(c));
}

// Short rows leave most of a block idle, many of them cost a block's start each: a wave
// per row up to 512 columns, and below 2048 from 4096 rows on (us, block / wave: [65536, 512]
// 52.4 / 23.0, [700, 512] 2.75 / 2.59, [8192, 1024] 10.9 / 8.1, [2048, 1024] 4.0 / 4.05,
// [8192, 1408] 11.9 / 10.5, [8192, 2048] 13.4 / 13.9).
template <bool SILU>
static void quant_fp8(hipStream_t st, const void* x, void* q, void* scales, int T, int K) {
#define QUANT(TPR)                                                                                  \
    hipLaunchKernelGGL((quant_fp8_kernel<SILU, TPR>), dim3(CEIL_DIV(T, 256 / TPR)), dim3(256), 0, st, \
                       (const uint4*)x, (uint2*)q, (float*)scales, T, K / 8)
    if (K <= 512 || (K < 2048 && T >= 4096)) QUANT(64);
    else QUANT(256);
#undef QUANT
}

extern "C" int oa_quant_fp8(void* stream, const void* x, void* q, void* scales,
                            int T, int K) {
    if (K % 8 != 0) return -100;
    quant_fp8<false>((hipStream_t)stream, x, q, scales, T, K);
    HIP_CHECK_LAUNCH();
    return 0;
}

// silu(gu[t, :K]) * gu[t, K:] of gu [T, 2 K], quantized
extern "C" int oa_silu_quant_fp8(void* stream, const void* gu, void* q, void* scales,
                                 int T, int K) {
    if (K % 8 != 0) return -100;
    if ((uintptr_t)gu % 16 != 0) return -101;
    quant_fp8<true>((hipStream_t)stream, gu, q, scales, T, K);
    HIP_CHECK_LAUNCH();
    return 0;
}

// ---- fp8-weight GEMV (decode path) -----------------------------------------
// out[M, N] = (x[M, K] @ W8[N, K]^T) * w_scale[n]; x bf16.
// NORM / ADDRES mirror the bf16 gemv fusions: rmsnorm prologue on x
// (fp32 rstd pass) and a residual-add epilogue.

// fp32 rstd of x row m (same as gemv.hip's row_rstd; separate TU)
__device__ __forceinline__ float row_rstd8(const uint32_t* xrow, int k2,
                                           int lane, float eps) {
    float ss = 0.0f;
    for (int i = lane * 4; i < k2; i += WAVE * 4) {
        uint4 xv = *reinterpret_cast<const uint4*>(xrow + i);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float lo = bf16_lo((&xv.x)[j]), hi = bf16_hi((&xv.x)[j]);
            ss = fmaf(lo, lo, ss);
            ss = fmaf(hi, hi, ss);
        }
    }
    ss = wave_reduce_sum(ss);
    return rsqrtf(ss / (float)(k2 * 2) + eps);
}

// XS: stage x as PRE-SCALED f32 in LDS once per block (requires M*K*4 <=
// 128 KiB). The fp8 dequant stream loop was VALU-bound at ~4.5 TB/s: per
// 16 W bytes it spent ~16 VALU unpacking the bf16 x (plus 4 more per
// element on the NORM path); the f32 image folds the rmsnorm weight and
// rstd in at fill time, leaving cvt+fma only in the stream loop.
// RW=2: two adjacent W rows per wave — the (expensive) bf16 x unpack
// amortizes over both fp8 streams, the same structure that makes the
// gateup form the fastest fp8 VALU stream (5.96 vs 5.1 TB/s measured).
template <int M, bool NORM, bool ADDRES, bool XS = false, int RW = 1>
__global__ __launch_bounds__(256) void gemv_fp8_kernel(
    const uint32_t* __restrict__ x,   // [M, K/2] bf16x2
    const uint32_t* __restrict__ w8,  // [N, K/4] fp8x4
    const float* __restrict__ wscale, // [N]
    uint32_t* __restrict__ out,       // [M, N] bf16
    const uint32_t* __restrict__ wn,  // [K/2] rmsnorm weight (NORM)
    const uint32_t* __restrict__ res, // [M, N] residual (ADDRES)
    int N, int K, float eps) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int wid = threadIdx.x / WAVE;
    const int k4 = K / 4;
    const int k2 = K / 2;

    float rstd[M];
    if (NORM) {
#pragma unroll
        for (int m = 0; m < M; ++m)
            rstd[m] = row_rstd8(x + (size_t)m * k2, k2, lane, eps);
    }

    extern __shared__ float xs[];  // [M][K] f32, XS only
    if (XS) {
        for (int idx = threadIdx.x; idx < M * k2; idx += blockDim.x) {
            const int m = idx / k2;
            const int i2 = idx % k2;  // word index in row
            const uint32_t xv = x[(size_t)m * k2 + i2];
            float lo = bf16_lo(xv), hi = bf16_hi(xv);
            if (NORM) {
                const uint32_t w = wn[i2];
                lo *= rstd[m] * bf16_lo(w);
                hi *= rstd[m] * bf16_hi(w);
            }
            xs[(size_t)m * K + i2 * 2] = lo;
            xs[(size_t)m * K + i2 * 2 + 1] = hi;
        }
        __syncthreads();
    }

    for (int row0 = (blockIdx.x * 4 + wid) * RW; row0 < N;
         row0 += gridDim.x * 4 * RW) {
        const uint32_t* wrow[RW];
        bool live[RW];
#pragma unroll
        for (int rr = 0; rr < RW; ++rr) {
            live[rr] = row0 + rr < N;
            wrow[rr] = w8 + (size_t)(live[rr] ? row0 + rr : row0) * k4;
        }
        float acc[RW][M];
#pragma unroll
        for (int rr = 0; rr < RW; ++rr)
#pragma unroll
            for (int m = 0; m < M; ++m) acc[rr][m] = 0.0f;
        // 16 B per lane = 16 fp8 elements per pass per row stream; the
        // bf16 x unpack happens ONCE and feeds every stream
        for (int i = lane * 4; i < k4; i += WAVE * 4) {
            float wf[RW][16];
#pragma unroll
            for (int rr = 0; rr < RW; ++rr) {
                u32x4 wv = nt_load4f(wrow[rr] + i);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    f32x2 lo = fp8x2_to_f32<false>(wv[j]);
                    f32x2 hi = fp8x2_to_f32<true>(wv[j]);
                    wf[rr][j * 4 + 0] = lo[0];
                    wf[rr][j * 4 + 1] = lo[1];
                    wf[rr][j * 4 + 2] = hi[0];
                    wf[rr][j * 4 + 3] = hi[1];
                }
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
                float xf[16];
                if (XS) {
                    const float* xr = xs + (size_t)m * K + i * 4;
#pragma unroll
                    for (int e = 0; e < 16; ++e) xf[e] = xr[e];
                } else {
                    // matching 16 bf16 of x = 2 x 16B loads
                    uint4 xv0 = *reinterpret_cast<const uint4*>(
                        x + (size_t)m * k2 + i * 2);
                    uint4 xv1 = *reinterpret_cast<const uint4*>(
                        x + (size_t)m * k2 + i * 2 + 4);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        float x0l = bf16_lo((&xv0.x)[j]),
                              x0h = bf16_hi((&xv0.x)[j]);
                        float x1l = bf16_lo((&xv1.x)[j]),
                              x1h = bf16_hi((&xv1.x)[j]);
                        if (NORM) {
                            const uint32_t w0 = wn[i * 2 + j];
                            const uint32_t w1 = wn[i * 2 + 4 + j];
                            x0l *= rstd[m] * bf16_lo(w0);
                            x0h *= rstd[m] * bf16_hi(w0);
                            x1l *= rstd[m] * bf16_lo(w1);
                            x1h *= rstd[m] * bf16_hi(w1);
                        }
                        xf[j * 2] = x0l;
                        xf[j * 2 + 1] = x0h;
                        xf[8 + j * 2] = x1l;
                        xf[8 + j * 2 + 1] = x1h;
                    }
                }
#pragma unroll
                for (int rr = 0; rr < RW; ++rr)
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        acc[rr][m] = fmaf(xf[e], wf[rr][e], acc[rr][m]);
            }
        }
#pragma unroll
        for (int rr = 0; rr < RW; ++rr) {
            const float sc = wscale[live[rr] ? row0 + rr : row0];
#pragma unroll
            for (int m = 0; m < M; ++m) {
                float v = wave_reduce_sum(acc[rr][m]) * sc;
                if (lane == 0 && live[rr]) {
                    if (ADDRES)
                        v += bf16_to_f32(reinterpret_cast<const uint16_t*>(
                            res)[(size_t)m * N + row0 + rr]);
                    reinterpret_cast<uint16_t*>(
                        out)[(size_t)m * N + row0 + rr] = f32_to_bf16(v);
                }
            }
        }
    }
}

// Fused fp8 gate-up + SiLU: fused weight holds gate rows [0, I) and up rows
// [I, 2I); each wave streams BOTH fp8 rows and writes silu(g)*u directly.
template <int M, bool NORM, bool XS = false>
__global__ __launch_bounds__(256) void gemv_gateup_fp8_kernel(
    const uint32_t* __restrict__ x, const uint32_t* __restrict__ w8,
    const float* __restrict__ wscale /* [2I] */, uint32_t* __restrict__ out,
    const uint32_t* __restrict__ wn, int I, int K, float eps) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int wid = threadIdx.x / WAVE;
    const int k4 = K / 4;
    const int k2 = K / 2;

    float rstd[M];
    if (NORM) {
#pragma unroll
        for (int m = 0; m < M; ++m)
            rstd[m] = row_rstd8(x + (size_t)m * k2, k2, lane, eps);
    }

    extern __shared__ float xs[];  // [M][K] f32, XS only (pre-scaled)
    if (XS) {
        for (int idx = threadIdx.x; idx < M * k2; idx += blockDim.x) {
            const int m = idx / k2;
            const int i2 = idx % k2;
            const uint32_t xv = x[(size_t)m * k2 + i2];
            float lo = bf16_lo(xv), hi = bf16_hi(xv);
            if (NORM) {
                const uint32_t w = wn[i2];
                lo *= rstd[m] * bf16_lo(w);
                hi *= rstd[m] * bf16_hi(w);
            }
            xs[(size_t)m * K + i2 * 2] = lo;
            xs[(size_t)m * K + i2 * 2 + 1] = hi;
        }
        __syncthreads();
    }

    // RW adjacent row-pairs per wave at M=1: 2*RW fp8 streams share ONE x
    // unpack per pass (the amortization that took the plain kernel to RW=2)
    constexpr int RW = (M == 1 && !XS) ? 2 : 1;
    for (int row0 = (blockIdx.x * 4 + wid) * RW; row0 < I;
         row0 += gridDim.x * 4 * RW) {
        bool liver[RW];
        const uint32_t* wgr[RW];
        const uint32_t* wur[RW];
#pragma unroll
        for (int rr = 0; rr < RW; ++rr) {
            liver[rr] = row0 + rr < I;
            const int r = liver[rr] ? row0 + rr : row0;
            wgr[rr] = w8 + (size_t)r * k4;
            wur[rr] = w8 + (size_t)(r + I) * k4;
        }
        float accg[RW][M], accu[RW][M];
#pragma unroll
        for (int rr = 0; rr < RW; ++rr)
#pragma unroll
            for (int m = 0; m < M; ++m) accg[rr][m] = accu[rr][m] = 0.0f;
        for (int i = lane * 4; i < k4; i += WAVE * 4) {
          if constexpr (RW == 2) {
            // M == 1 here: unpack x ONCE, feed all four fp8 streams
            uint4 xv0 = *reinterpret_cast<const uint4*>(x + i * 2);
            uint4 xv1 = *reinterpret_cast<const uint4*>(x + i * 2 + 4);
            float xf[16];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float x0l = bf16_lo((&xv0.x)[j]), x0h = bf16_hi((&xv0.x)[j]);
                float x1l = bf16_lo((&xv1.x)[j]), x1h = bf16_hi((&xv1.x)[j]);
                if (NORM) {
                    const uint32_t w0 = wn[i * 2 + j];
                    const uint32_t w1 = wn[i * 2 + 4 + j];
                    x0l *= rstd[0] * bf16_lo(w0);
                    x0h *= rstd[0] * bf16_hi(w0);
                    x1l *= rstd[0] * bf16_lo(w1);
                    x1h *= rstd[0] * bf16_hi(w1);
                }
                xf[j * 2] = x0l;
                xf[j * 2 + 1] = x0h;
                xf[8 + j * 2] = x1l;
                xf[8 + j * 2 + 1] = x1h;
            }
#pragma unroll
            for (int rr = 0; rr < RW; ++rr) {
                u32x4 wvg = nt_load4f(wgr[rr] + i);
                u32x4 wvu = nt_load4f(wur[rr] + i);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    f32x2 gl = fp8x2_to_f32<false>(wvg[j]);
                    f32x2 gh = fp8x2_to_f32<true>(wvg[j]);
                    f32x2 ul = fp8x2_to_f32<false>(wvu[j]);
                    f32x2 uh = fp8x2_to_f32<true>(wvu[j]);
                    accg[rr][0] = fmaf(xf[j * 4 + 0], gl[0], accg[rr][0]);
                    accg[rr][0] = fmaf(xf[j * 4 + 1], gl[1], accg[rr][0]);
                    accg[rr][0] = fmaf(xf[j * 4 + 2], gh[0], accg[rr][0]);
                    accg[rr][0] = fmaf(xf[j * 4 + 3], gh[1], accg[rr][0]);
                    accu[rr][0] = fmaf(xf[j * 4 + 0], ul[0], accu[rr][0]);
                    accu[rr][0] = fmaf(xf[j * 4 + 1], ul[1], accu[rr][0]);
                    accu[rr][0] = fmaf(xf[j * 4 + 2], uh[0], accu[rr][0]);
                    accu[rr][0] = fmaf(xf[j * 4 + 3], uh[1], accu[rr][0]);
                }
            }
            continue;
          }

            u32x4 wvg = nt_load4f(wgr[0] + i);
            u32x4 wvu = nt_load4f(wur[0] + i);
            float wfg[16], wfu[16];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                f32x2 gl = fp8x2_to_f32<false>(wvg[j]);
                f32x2 gh = fp8x2_to_f32<true>(wvg[j]);
                f32x2 ul = fp8x2_to_f32<false>(wvu[j]);
                f32x2 uh = fp8x2_to_f32<true>(wvu[j]);
                wfg[j * 4 + 0] = gl[0]; wfg[j * 4 + 1] = gl[1];
                wfg[j * 4 + 2] = gh[0]; wfg[j * 4 + 3] = gh[1];
                wfu[j * 4 + 0] = ul[0]; wfu[j * 4 + 1] = ul[1];
                wfu[j * 4 + 2] = uh[0]; wfu[j * 4 + 3] = uh[1];
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
                if (XS) {
                    const float* xr = xs + (size_t)m * K + i * 4;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        float4 a = *reinterpret_cast<const float4*>(xr + q * 4);
                        accg[0][m] = fmaf(a.x, wfg[q * 4 + 0], accg[0][m]);
                        accg[0][m] = fmaf(a.y, wfg[q * 4 + 1], accg[0][m]);
                        accg[0][m] = fmaf(a.z, wfg[q * 4 + 2], accg[0][m]);
                        accg[0][m] = fmaf(a.w, wfg[q * 4 + 3], accg[0][m]);
                        accu[0][m] = fmaf(a.x, wfu[q * 4 + 0], accu[0][m]);
                        accu[0][m] = fmaf(a.y, wfu[q * 4 + 1], accu[0][m]);
                        accu[0][m] = fmaf(a.z, wfu[q * 4 + 2], accu[0][m]);
                        accu[0][m] = fmaf(a.w, wfu[q * 4 + 3], accu[0][m]);
                    }
                    continue;
                }
                uint4 xv0 = *reinterpret_cast<const uint4*>(x + (size_t)m * k2 + i * 2);
                uint4 xv1 = *reinterpret_cast<const uint4*>(x + (size_t)m * k2 + i * 2 + 4);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float x0l = bf16_lo((&xv0.x)[j]), x0h = bf16_hi((&xv0.x)[j]);
                    float x1l = bf16_lo((&xv1.x)[j]), x1h = bf16_hi((&xv1.x)[j]);
                    if (NORM) {
                        const uint32_t w0 = wn[i * 2 + j];
                        const uint32_t w1 = wn[i * 2 + 4 + j];
                        x0l *= rstd[m] * bf16_lo(w0);
                        x0h *= rstd[m] * bf16_hi(w0);
                        x1l *= rstd[m] * bf16_lo(w1);
                        x1h *= rstd[m] * bf16_hi(w1);
                    }
                    accg[0][m] = fmaf(x0l, wfg[j * 2], accg[0][m]);
                    accg[0][m] = fmaf(x0h, wfg[j * 2 + 1], accg[0][m]);
                    accg[0][m] = fmaf(x1l, wfg[8 + j * 2], accg[0][m]);
                    accg[0][m] = fmaf(x1h, wfg[8 + j * 2 + 1], accg[0][m]);
                    accu[0][m] = fmaf(x0l, wfu[j * 2], accu[0][m]);
                    accu[0][m] = fmaf(x0h, wfu[j * 2 + 1], accu[0][m]);
                    accu[0][m] = fmaf(x1l, wfu[8 + j * 2], accu[0][m]);
                    accu[0][m] = fmaf(x1h, wfu[8 + j * 2 + 1], accu[0][m]);
                }
            }
        }
#pragma unroll
        for (int rr = 0; rr < RW; ++rr) {
            const int row = liver[rr] ? row0 + rr : row0;
            const float sg = wscale[row], su = wscale[row + I];
#pragma unroll
            for (int m = 0; m < M; ++m) {
                float g = wave_reduce_sum(accg[rr][m]) * sg;
                float u = wave_reduce_sum(accu[rr][m]) * su;
                if (lane == 0 && liver[rr]) {
                    const float act = g / (1.0f + __expf(-g)) * u;
                    reinterpret_cast<uint16_t*>(out)[(size_t)m * I + row] =
                        f32_to_bf16(act);
                }
            }
        }
    }
}

// mode: 0 plain, 1 norm-prologue, 2 residual-add epilogue, 3 both
extern "C" int oa_gemv_fp8_mfma(void* stream, const void* x, const void* w8,
                                const void* wscale, void* out, const void* wn,
                                const void* res, int M, int N, int K,
                                float eps, int mode, int gateup);

// MFMA path eligibility (see the v3 kernel at the end of this file).
// A/B-measured (profiles/README.md, scripts/gemv_fp8_bench.py): the MFMA
// stream wins for M >= 2 (batched decode: +45..+59% at M=4 — the extra
// batch columns ride the same weight stream for free) while the VALU
// kernel's contiguous row-per-wave streams stay ahead at M=1 (5.1 vs 3.1
// TB/s: 16 strided row streams per wave + the x-quant launch don't pay off
// for one column). OPSAGENT_FP8_GEMV_MFMA=0 forces VALU, =2 forces MFMA.
static bool gemv_fp8_use_mfma(int M, int rows, int K, int gateup) {
    const char* e = getenv("OPSAGENT_FP8_GEMV_MFMA");
    if (e && e[0] == '0') return false;
    // must mirror oa_gemv_fp8_mfma's guards exactly (PF-deep prefetch ring
    // needs (K/512) % PF == 0) so ineligible shapes FALL BACK, not error
    if (K % 512 != 0 || (K / 512) % (gateup ? 4 : 8) != 0 || K > 32768 ||
        M > 16)
        return false;
    if (M < 2 && !(e && e[0] == '2')) return false;
    (void)rows;
    return (size_t)M * K <= 128 * 1024;
}

// One activation row, K a multiple of 2048 up to 16384: the scheme of the bf16 one-row
// kernel (gemv.hip) on fp8 weights. The block's activations, normalised there with NORM,
// are a float32 image in LDS, made once while the first weights are under way, four
// planes of four columns in sixteen so that a wave's 16-byte reads are contiguous; a wave
// streams the rows of its units, every waves-th of the weight, two at a time (GU: a gate
// row and its up row) in groups
// of GR 1024-column chunks, the next group under way while one is in use. us inside a
// decode step, the forms above with their normalisation in a launch of its own / here:
// gate-up 2 x 14336 x 4096 27.4 / 21.9, 6144 x 4096 11.1 / 7.8, 4096 x 14336 13.5 / 12.1;
// asking for the activations before the weights is 3 us of the normalised ones. A third
// group under way from the start cost more in waits than it hid (gate-up 27.6), seven
// chunks a group too (4096 x 14336 14.0).
template <bool NORM, bool ADDRES, bool GU, int GR, int XV, int WV>
__global__ __launch_bounds__(WV * 64) void gemv1_fp8_kernel(
    const uint4* __restrict__ x, const uint32_t* __restrict__ w8, const float* __restrict__ wscale,
    uint16_t* __restrict__ out, const uint4* __restrict__ wn, const uint16_t* __restrict__ res,
    int N, int K, int waves, int full, int extra, float eps) {
    extern __shared__ __attribute__((aligned(16))) float xl[];   // [4][K / 4]
    __shared__ float part[8];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int units = GU ? N : N / 2;
    const int u0 = blockIdx.x * WV + wid;
    const int k4 = K / 4, groups = K / (1024 * GR);
    const int total = (full + (u0 < extra)) * groups;       // of every waves-th unit
    auto row_of = [&](int u, int t) { return GU ? u + t * N : u * 2 + t; };
    u32x4 a[GR][2], b[GR][2];
    int u = min(u0, units - 1), g = 0;                      // of the group loaded last
    auto load = [&](u32x4 (&v)[GR][2]) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < GR; ++i)
                v[i][t] = nt_load4f(w8 + (size_t)row_of(u, t) * k4 + (g * GR + i) * 256 + lane * 4);
    };
    auto next = [&](u32x4 (&v)[GR][2]) {
        if (++g == groups) {
            g = 0;
            u += waves;
        }
        load(v);
        __builtin_amdgcn_sched_barrier(0);
    };
    // Loads return in order: the activations and lane i's scale and residual of the wave's
    // unit i (per <= 64) are asked for before the weights, so that the image below waits
    // for them alone.
    uint4 xv[XV], nv[XV];
#pragma unroll
    for (int j = 0; j < XV; ++j) {
        const int i = min(j * WV * 64 + tid, K / 8 - 1);
        xv[j] = x[i];
        if (NORM) nv[j] = wn[i];
    }
    float sc[2], rs[2] = {0.0f, 0.0f};
    {
        const int mine = (int)min(u0 + lane * (int64_t)waves, units - (int64_t)1);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            sc[t] = wscale[row_of(mine, t)];
            if (ADDRES) rs[t] = bf16_to_f32(res[row_of(mine, t)]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    load(a);
    __builtin_amdgcn_sched_barrier(0);

    float rstd = 1.0f;
    if (NORM) {
        // the sum of squares in one order however many waves share a row of 4096
        constexpr int SP = WV == 4 ? XV : 1;
#pragma unroll
        for (int p = 0; p < SP; ++p) {
            float ss = 0.0f;
#pragma unroll
            for (int j = p; j < (SP == 1 ? XV : p + 1); ++j)
                if (j * WV * 64 + tid < K / 8)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float lo = bf16_lo((&xv[j].x)[e]), hi = bf16_hi((&xv[j].x)[e]);
                        ss = fmaf(lo, lo, ss);
                        ss = fmaf(hi, hi, ss);
                    }
            ss = wave_reduce_sum(ss);
            if (lane == 0) part[p * WV + wid] = ss;
        }
        __syncthreads();
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < SP * WV; ++i) ss += part[i];
        rstd = rsqrtf(ss / (float)K + eps);
    }
#pragma unroll
    for (int j = 0; j < XV; ++j) {
        const int i = j * WV * 64 + tid;                        // columns i * 8 .. + 7
        if (i >= K / 8) continue;
        float f[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            f[2 * e] = bf16_lo((&xv[j].x)[e]);
            f[2 * e + 1] = bf16_hi((&xv[j].x)[e]);
            if (NORM) {
                f[2 * e] *= rstd * bf16_lo((&nv[j].x)[e]);
                f[2 * e + 1] *= rstd * bf16_hi((&nv[j].x)[e]);
            }
        }
        float* at = xl + (i & 1) * 2 * k4 + (i >> 1) * 4;
        *reinterpret_cast<float4*>(at) = make_float4(f[0], f[1], f[2], f[3]);
        *reinterpret_cast<float4*>(at + k4) = make_float4(f[4], f[5], f[6], f[7]);
    }
    __syncthreads();

    float acc[2] = {0.0f, 0.0f};
    int uu = 0, ug = 0;                                     // unit of the wave, group in use
    auto use = [&](u32x4 (&v)[GR][2]) {
#pragma unroll
        for (int i = 0; i < GR; ++i) {
            const int c = (ug * GR + i) * 64 + lane;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 f = reinterpret_cast<const float4*>(xl + q * k4)[c];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const f32x2 lo = fp8x2_to_f32<false>(v[i][t][q]), hi = fp8x2_to_f32<true>(v[i][t][q]);
                    float d = acc[t];
                    d = fmaf(f.x, lo[0], d);
                    d = fmaf(f.y, lo[1], d);
                    d = fmaf(f.z, hi[0], d);
                    acc[t] = fmaf(f.w, hi[1], d);
                }
            }
        }
        if (++ug == groups) {
            float r[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                r[t] = wave_reduce_sum(acc[t]) * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sc[t]), uu));
                if (ADDRES) r[t] += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rs[t]), uu));
                acc[t] = 0.0f;
            }
            if (lane == 0) {
                if (GU) out[u0 + uu * waves] = f32_to_bf16(r[0] / (1.0f + __expf(-r[0])) * r[1]);
                else reinterpret_cast<uint32_t*>(out)[u0 + uu * waves] = pack_bf16x2(r[0], r[1]);
            }
            ug = 0;
            ++uu;
        }
    };
    // the last groups are apart, so that every wait counts the loads behind it exactly
    int n = 0;
    for (; n + 2 < total; n += 2) {
        next(b);
        use(a);
        next(a);
        use(b);
    }
    if (n + 2 == total) {
        next(b);
        use(a);
        use(b);
    } else if (n < total) {
        use(a);
    }
}

static bool gemv1_fp8_ok(const void* x, const void* w8, const void* wn, const void* out, int M, int N,
                         int K, bool gateup) {
    return M == 1 && K % 2048 == 0 && K >= 2048 && K <= 16384 && N >= 1 && (gateup || N % 2 == 0) &&
           ((uintptr_t)x | (uintptr_t)w8 | (uintptr_t)wn) % 16 == 0 && (uintptr_t)out % 4 == 0;
}

// mode: 1 normalise x first, 2 add res
static int gemv1_fp8(hipStream_t st, const void* x, const void* w8, const void* wscale, void* out,
                     const void* wn, const void* res, int N, int K, float eps, int mode, bool gateup) {
    const int units = gateup ? N : N / 2;
    // As in gemv.hip: up to K = 4096 blocks of four waves of a unit each, no more than 32
    // blocks per CU (us, blocks of eight / this: 6144 x 4096 8.2 / 7.1, 4096 x 4096 6.5 / 5.8,
    // 28672 x 4096 22.2 / 21.1, 2 x 14336 x 4096 22.3 / 20.8, 5632 x 2048 4.9 / 4.9). Above: as
    // many blocks of eight waves as stay resident (two per CU), fewer and fuller ones where
    // that evens out the CUs by more than a fifth.
    const int wv = K <= 4096 ? 4 : 8;
    int per = CEIL_DIV(units, wv == 4 ? 256 * 4 * 32 : 256 * 8 * 2);
    if (wv == 8) {
        auto rounds = [&](int p) { return CEIL_DIV(CEIL_DIV(CEIL_DIV(units, p), 8), 256) * p; };
        for (int p = per + 1, p1 = 2 * per + 1; p <= p1; ++p)
            if (rounds(p) * 5 < rounds(per) * 4) per = p;
    }
    if (per > 64) per = 64;
    const int blocks = CEIL_DIV(CEIL_DIV(units, per), wv);
    const int waves = blocks * wv;
#define G1F(NV, RV, GV, GR, XV, WV)                                                                   \
    hipLaunchKernelGGL((gemv1_fp8_kernel<NV, RV, GV, GR, XV, WV>), dim3(blocks), dim3(WV * 64), (size_t)K * 4, \
                       st, (const uint4*)x, (const uint32_t*)w8, (const float*)wscale,                \
                       (uint16_t*)out, (const uint4*)wn, (const uint16_t*)res, N, K, waves,           \
                       units / waves, units % waves, eps)
#define G1FK(NV, RV, GV)                                \
    do {                                                \
        if (K == 4096) G1F(NV, RV, GV, 4, 2, 4);        \
        else if (K < 4096) G1F(NV, RV, GV, 2, 1, 4);    \
        else G1F(NV, RV, GV, 2, 4, 8);                  \
    } while (0)
    if (gateup) {
        if (mode & 1) G1FK(true, false, true);
        else G1FK(false, false, true);
    } else {
        switch (mode) {
            case 0: G1FK(false, false, false); break;
            case 1: G1FK(true, false, false); break;
            case 2: G1FK(false, true, false); break;
            case 3: G1FK(true, true, false); break;
            default: return -102;
        }
    }
#undef G1FK
#undef G1F
    HIP_CHECK_LAUNCH();
    return 0;
}

extern "C" int oa_gemv_fp8_ex(void* stream, const void* x, const void* w8,
                              const void* wscale, void* out, const void* wn,
                              const void* res, int M, int N, int K, float eps,
                              int mode) {
    if (K % 16 != 0) return -100;
    if (gemv_fp8_use_mfma(M, N, K, 0))
        return oa_gemv_fp8_mfma(stream, x, w8, wscale, out, wn, res, M, N, K,
                                eps, mode, 0);
    if (gemv1_fp8_ok(x, w8, mode & 1 ? wn : nullptr, out, M, N, K, false))
        return gemv1_fp8((hipStream_t)stream, x, w8, wscale, out, wn, res, N, K, eps, mode, false);
    // M=1 runs the RW=2 two-stream form (x unpack amortized — the gateup
    // structure measured 5.96 vs 5.1 TB/s); OPSAGENT_FP8_GEMV_RW=1 forces
    // the single-stream form for A/B.
    const char* rwe = getenv("OPSAGENT_FP8_GEMV_RW");
    const int rw = (M == 1 && !(rwe && rwe[0] == '1')) ? 2 : 1;
    const int grid = min(4096, CEIL_DIV(N, 4 * rw));
    // pre-scaled f32 x image in LDS: measured NET NEGATIVE on the 70B fp8
    // turn (747 vs 503 ms — the 32-114 KiB LDS footprint collapses block
    // occupancy, which this latency-hiding structure needs more than the
    // saved unpack VALU). Default OFF; OPSAGENT_FP8_GEMV_XS=1 re-enables
    // for A/B.
    const size_t xs_bytes = (size_t)M * K * 4;
    const char* xse = getenv("OPSAGENT_FP8_GEMV_XS");
    const bool use_xs = xs_bytes <= 131072 && xse && xse[0] == '1';
#define LAUNCH_F8NM(MV, NORMV, RESV)                                           \
    do {                                                                       \
        if (use_xs)                                                            \
            hipLaunchKernelGGL((gemv_fp8_kernel<MV, NORMV, RESV, true>),       \
                               dim3(grid), dim3(256), xs_bytes,                \
                               (hipStream_t)stream, (const uint32_t*)x,        \
                               (const uint32_t*)w8, (const float*)wscale,      \
                               (uint32_t*)out, (const uint32_t*)wn,            \
                               (const uint32_t*)res, N, K, eps);               \
        else if (rw == 2)                                                      \
            hipLaunchKernelGGL(                                                \
                (gemv_fp8_kernel<MV, NORMV, RESV, false, 2>), dim3(grid),      \
                dim3(256), 0, (hipStream_t)stream, (const uint32_t*)x,         \
                (const uint32_t*)w8, (const float*)wscale, (uint32_t*)out,     \
                (const uint32_t*)wn, (const uint32_t*)res, N, K, eps);         \
        else                                                                   \
            hipLaunchKernelGGL((gemv_fp8_kernel<MV, NORMV, RESV, false>),      \
                               dim3(grid), dim3(256), 0, (hipStream_t)stream,  \
                               (const uint32_t*)x, (const uint32_t*)w8,        \
                               (const float*)wscale, (uint32_t*)out,           \
                               (const uint32_t*)wn, (const uint32_t*)res, N,   \
                               K, eps);                                        \
    } while (0)
#define LAUNCH_F8(MV)                                                          \
    do {                                                                       \
        switch (mode) {                                                        \
            case 0: LAUNCH_F8NM(MV, false, false); break;                      \
            case 1: LAUNCH_F8NM(MV, true, false); break;                       \
            case 2: LAUNCH_F8NM(MV, false, true); break;                       \
            case 3: LAUNCH_F8NM(MV, true, true); break;                        \
            default: return -102;                                              \
        }                                                                      \
    } while (0)
    switch (M) {
        case 1: LAUNCH_F8(1); break;
        case 2: LAUNCH_F8(2); break;
        case 3: LAUNCH_F8(3); break;
        case 4: LAUNCH_F8(4); break;
        case 5: LAUNCH_F8(5); break;
        case 6: LAUNCH_F8(6); break;
        case 7: LAUNCH_F8(7); break;
        case 8: LAUNCH_F8(8); break;
        case 12: LAUNCH_F8(12); break;
        case 16: LAUNCH_F8(16); break;
        default: return -101;
    }
#undef LAUNCH_F8
#undef LAUNCH_F8NM
    HIP_CHECK_LAUNCH();
    return 0;
}

extern "C" int oa_gemv_fp8(void* stream, const void* x, const void* w8,
                           const void* wscale, void* out, int M, int N, int K) {
    return oa_gemv_fp8_ex(stream, x, w8, wscale, out, nullptr, nullptr, M, N,
                          K, 0.0f, 0);
}

extern "C" int oa_gemv_gateup_fp8(void* stream, const void* x, const void* w8,
                                  const void* wscale, void* out,
                                  const void* wn, int M, int I, int K,
                                  float eps, int norm) {
    if (K % 16 != 0) return -100;
    if (gemv_fp8_use_mfma(M, I, K, 1))
        return oa_gemv_fp8_mfma(stream, x, w8, wscale, out, wn, nullptr, M,
                                2 * I, K, eps, norm ? 1 : 0, 1);
    if (gemv1_fp8_ok(x, w8, norm ? wn : nullptr, out, M, I, K, true))
        return gemv1_fp8((hipStream_t)stream, x, w8, wscale, out, wn, nullptr, I, K, eps, norm ? 1 : 0,
                         true);
    // M=1 instantiates RW=2 row-pairs (4 streams/wave)
    const int grid = min(4096, CEIL_DIV(I, M == 1 ? 8 : 4));
    const size_t xs_bytes = (size_t)M * K * 4;
    const char* xse = getenv("OPSAGENT_FP8_GEMV_XS");
    const bool use_xs = xs_bytes <= 131072 && xse && xse[0] == '1';
#define LAUNCH_GU8_1(MV, NORMV, XSV, SH)                                       \
    hipLaunchKernelGGL((gemv_gateup_fp8_kernel<MV, NORMV, XSV>), dim3(grid),   \
                       dim3(256), SH, (hipStream_t)stream,                     \
                       (const uint32_t*)x, (const uint32_t*)w8,                \
                       (const float*)wscale, (uint32_t*)out,                   \
                       (const uint32_t*)wn, I, K, eps)
#define LAUNCH_GU8(MV)                                                         \
    do {                                                                       \
        if (norm) {                                                            \
            if (use_xs) LAUNCH_GU8_1(MV, true, true, xs_bytes);                \
            else LAUNCH_GU8_1(MV, true, false, 0);                             \
        } else {                                                               \
            if (use_xs) LAUNCH_GU8_1(MV, false, true, xs_bytes);               \
            else LAUNCH_GU8_1(MV, false, false, 0);                            \
        }                                                                      \
    } while (0)
    switch (M) {
        case 1: LAUNCH_GU8(1); break;
        case 2: LAUNCH_GU8(2); break;
        case 3: LAUNCH_GU8(3); break;
        case 4: LAUNCH_GU8(4); break;
        case 6: LAUNCH_GU8(6); break;
        case 8: LAUNCH_GU8(8); break;
        default: return -101;
    }
#undef LAUNCH_GU8
#undef LAUNCH_GU8_1
    HIP_CHECK_LAUNCH();
    return 0;
}

// ---- fp8 MFMA tile GEMM (prefill path) -------------------------------------
// C[M, N] = (A8[M, K] @ B8[N, K]^T) * a_scale[m] * b_scale[n], bf16 out.
//
// A tile of BM x BN, sixteen waves (4 x 4; 96 rows: fourteen, 3 x 4 and two), K-steps of 128 fp8 bytes, A and B staged by
// 16-byte global_load_lds. 16-byte chunk c of row r lies at c ^ (r >> 1 & 7): LDS has 64
// banks, and 16 rows of 128 bytes at one chunk touch each of them once (c ^ (r & 7) touches
// half of them twice: 11 M conflict cycles of 22 M on 28672 x 4096, M = 700, none here). The
// swizzle is on the source address, as the transfer writes lanes in order. Rows past M or N
// repeat the last one and are not stored.
//
// The products are v_mfma_scale_f32_32x32x64_f8f6f4 with identity E8M0 scales (0x7f =
// 2^0): the large-K scaled forms are the only fp8 MFMAs past the bf16 rate on gfx950;
// with unit scales the numerics are plain fp8 products with float32 accumulation.
// Fragment maps: A lane l & 31 = row, l >> 5 = 32-byte k-half; B the same over columns.

typedef __attribute__((ext_vector_type(8))) int i32x8_f8;   // 32 fp8 (MX operand)
typedef __attribute__((ext_vector_type(16))) float f32x16_t;  // 32x32 C/D

#define GK2 128   // K step in fp8 bytes

template <int V>
__device__ __forceinline__ void g8_wait() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(V) : "memory");
}

// A ring of ST K-steps: ST - 1 are under way while one is in use. A wait leaves the younger
// steps' transfers in flight (vmcnt counts them in order); the barrier after it says both
// that step t has landed for every wave and that step t - 1 is no longer read, so its
// buffer can be filled. The transfers are inline asm because hipcc's wait inserter drains
// builtin ones before the first LDS read. Work items go to the dies in runs, with the row
// tiles of a column strip next to each other: a strip is read into one die's L2 once.
//
// What bounds it is how well the waves of a CU cover each other's waits at the barrier and
// for fragments: the matrix cores are busy for a third of the time, the LDS for a sixth, and
// the L2 gives a CU 50 GB/s of the 150 it can. Hence sixteen waves, however small their part:
// 4096 x 4096, M = 700 29.3 us with four waves, 23.5 with eight, 21.1 with sixteen; 4096 x
// 14336 75 / 64 / 60; 28672 x 4096 in tiles of 128 x 256 114 with eight, 108 with sixteen.
// Reading fragments ahead of the products, carrying them over the barrier and spreading the
// transfers between the products were all slower. us, before (128 x 128, four waves) / 128 x
// 128 in a ring of four / two blocks a CU in rings of two / 128 x 256 in three / 256 x 256 in
// two: 28672 x 4096, M = 512 94 / 96 / 85 / 78 / 68, 700 128 / 130 / 119 / 108 / 119, 2048 306 /
// 331 / 290 / 271 / 251; 4096 x 14336, 700 76 / 61 / 101 / 94 / 162, 2048 132 / 146 / 139 / 112 /
// 173; 6144 x 4096, 700 34.5 / 40.5 / 30.1 / 31.8 / 49; 2048 x 8192, 700 45.9 / 33.7 / 43 / 49 /
// 81; 16384 x 2048, 700 52.9 / 43.5 / 42.9 / 44.2 / 37.9.
#define G8_WAVES(BM) ((BM) == 96 ? 14 : 16)
template <int BM, int BN, int ST, int BLOCKS>
__global__ __launch_bounds__(64 * G8_WAVES(BM), 4 * BLOCKS) void gemm_fp8_tile_kernel(
    const char* __restrict__ a8, const char* __restrict__ b8,
    const float* __restrict__ ascale, const float* __restrict__ bscale,
    uint16_t* __restrict__ c, int M, int N, int K, int mtiles, int items) {
    constexpr int FI = BM == 96 ? 1 : BM / 128, FJ = BN / 128;         // fragments of a wave
    constexpr int WAVES = G8_WAVES(BM);
    constexpr int STEP = (BM + BN) * GK2, LPW = (BM + BN) / (8 * WAVES);     // transfers of a wave
    static_assert(LPW * WAVES * 8 == BM + BN, "every wave transfers as much");
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int per = gridDim.x >> 3;
    const int item = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (item >= items) return;
    const int nt = item / mtiles;
    const int tm = (item - nt * mtiles) * BM, tn = nt * BN;
    const int lane = threadIdx.x & (WAVE - 1);
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int wr = wid >> 2, wc = wid & 3;

    const char* src[LPW];
#pragma unroll
    for (int p = 0; p < LPW; ++p) {
        const int r = (p * WAVES + wid) * 8 + (lane >> 3);   // row of A, then of B
        const int64_t at = r < BM ? (int64_t)min(tm + r, M - 1) * K : (int64_t)min(tn + r - BM, N - 1) * K;
        src[p] = (r < BM ? a8 : b8) + at + ((lane & 7) ^ (r >> 1 & 7)) * 16;
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem + wid * 1024);
    auto stage = [&](int buf) {
#pragma unroll
        for (int p = 0; p < LPW; ++p) {
            lds_transfer16(lds0 + buf * STEP + p * WAVES * 1024, src[p]);
            src[p] += GK2;
        }
    };
    const int fr = lane & 31, kh = lane >> 5, sw = fr >> 1 & 7;
    auto frag = [&](const char* rows, int kk) {
        union {
            uint4 h[2];
            i32x8_f8 v;
        } f;
        f.h[0] = *reinterpret_cast<const uint4*>(rows + fr * GK2 + (((kk * 4 + kh * 2) ^ sw) << 4));
        f.h[1] = *reinterpret_cast<const uint4*>(rows + fr * GK2 + (((kk * 4 + kh * 2 + 1) ^ sw) << 4));
        return f.v;
    };
    f32x16_t acc[FI][FJ] = {};
    const int ns = K / GK2;
#pragma unroll
    for (int t = 0; t < ST - 1; ++t)
        if (t < ns) stage(t);
    int buf = 0;
    for (int t = 0; t < ns; ++t) {
        const int behind = min(ST - 2, ns - 1 - t);          // younger steps under way
        if (ST > 3 && behind >= 2) g8_wait<2 * LPW>();
        else if (ST > 2 && behind >= 1) g8_wait<LPW>();
        else g8_wait<0>();
        const char* ab = smem + buf * STEP + wr * FI * 32 * GK2;
        const char* bb = smem + buf * STEP + (BM + wc * FJ * 32) * GK2;
        if (t + ST - 1 < ns) stage(buf == 0 ? ST - 1 : buf - 1);
        if (wr * FI * 32 < BM)                               // (96 rows: two waves transfer alone)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            i32x8_f8 fa[FI], fb[FJ];
#pragma unroll
            for (int i = 0; i < FI; ++i) fa[i] = frag(ab + i * 32 * GK2, kk);
#pragma unroll
            for (int j = 0; j < FJ; ++j) fb[j] = frag(bb + j * 32 * GK2, kk);
#pragma unroll
            for (int i = 0; i < FI; ++i)
#pragma unroll
                for (int j = 0; j < FJ; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                        fa[i], fb[j], acc[i][j], 0, 0, 0, 0x7f, 0, 0x7f);
        }
        buf = buf + 1 == ST ? 0 : buf + 1;
    }

    if (wr * FI * 32 >= BM) return;
    // 32x32 C/D map: col = lane & 31, row = (r & 3) + 8 * (r >> 2) + 4 * (lane >> 5).
    // Row scales are read together (rows past the end repeat the last), not one by one
    // behind a branch each.
#pragma unroll
    for (int i = 0; i < FI; ++i) {
        const int row0 = tm + (wr * FI + i) * 32 + 4 * kh;
        float as[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) as[r] = ascale[min(row0 + (r & 3) + 8 * (r >> 2), M - 1)];
#pragma unroll
        for (int j = 0; j < FJ; ++j) {
            const int col = tn + (wc * FJ + j) * 32 + fr;
            if (col >= N) continue;
            const float bs = bscale[col];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = row0 + (r & 3) + 8 * (r >> 2);
                if (row < M) c[(size_t)row * N + col] = f32_to_bf16(acc[i][j][r] * as[r] * bs);
            }
        }
    }
}

// Tile by the rounds that the tiles take over 256 CUs, in the time of a step in us (figures
// above): one block of 128 x 128 a CU 0.62 (0.65 over several rounds, which start and end
// bare), two of them 1.27 and less where the second ones are few, 128 x 256 1.12, 256 x 256
// 1.9. It names the fastest for 39 of 40 sizes (12288 x 4096, M = 512: 42.1, 38.2).
//
// Tiles of 96 x 128, twelve waves at work and two that only transfer, take 0.54: the form where they fit one
// round, which 128 rows leave a quarter empty or filled with rows past the end. us, 128 / 96 rows a tile: 4096 x
// 14336, M = 300 55.6 / 49.6, 512 66.7 / 56.6, 700 68.9 / 59.4, 768 67.4 / 60.7; 4096 x 4096, 700 22.8 / 20.4;
// 2048 x 8192, 1400 38.5 / 33.6; but in two rounds 4096 x 14336, 1000 70.5 / 103.9, 2048 112 / 167.
static int gemm_fp8_tile(int64_t M, int64_t N, double* us = nullptr, int64_t* rounds = nullptr) {
    const int64_t n1 = CEIL_DIV(M, 128) * CEIL_DIV(N, 128), rest = n1 % 512;
    const int64_t n2 = CEIL_DIV(M, 128) * CEIL_DIV(N, 256), n3 = CEIL_DIV(M, 256) * CEIL_DIV(N, 256);
    const int64_t n4 = CEIL_DIV(M, 96) * CEIL_DIV(N, 128);
    const double t[5] = {n1 <= 256 ? 0.62 : CEIL_DIV(n1, 256) * 0.65,
                         n1 / 512 * 1.27 + (rest > 256 ? 0.86 + (rest - 256) * 0.0015 : rest > 0 ? 0.75 : 0.0),
                         CEIL_DIV(n2, 256) * 1.12, CEIL_DIV(n3, 256) * 1.9, n4 <= 256 ? 0.54 : 1e9};
    int best = 0;
    for (int i = 1; i < 5; ++i)
        if (t[i] < t[best]) best = i;
    if (us) *us = t[best];
    if (rounds) *rounds = best == 1 ? CEIL_DIV(n1, 512) : CEIL_DIV(best == 0 ? n1 : best == 2 ? n2 : best == 3 ? n3 : n4, 256);
    return best;
}

// its time, us: of the steps, and to start and to end each round (11% rms over 50 sizes)
extern "C" double oa_gemm_fp8_us(int M, int N, int K) {
    double us;
    int64_t rounds;
    gemm_fp8_tile(M, N, &us, &rounds);
    return 0.93 * us * (K / GK2) + 4.9 * rounds + 0.3;
}

extern "C" int oa_gemm_fp8(void* stream, const void* a8, const void* b8,
                           const void* ascale, const void* bscale, void* c,
                           int M, int N, int K) {
    if (K % GK2 != 0 || M < 1 || N < 1) return -100;
#define G8(BM, BN, ST, BLOCKS)                                                                     \
    do {                                                                                           \
        const int mt = CEIL_DIV(M, BM);                                                            \
        const int64_t items = (int64_t)CEIL_DIV(N, BN) * mt;                                       \
        if (items > (1 << 28)) return -101;                                                        \
        hipLaunchKernelGGL((gemm_fp8_tile_kernel<BM, BN, ST, BLOCKS>),                             \
                           dim3((unsigned)(CEIL_DIV(items, 8) * 8)), dim3(64 * G8_WAVES(BM)),      \
                           (ST) * (BM + BN) * GK2, (hipStream_t)stream, (const char*)a8,           \
                           (const char*)b8, (const float*)ascale, (const float*)bscale,            \
                           (uint16_t*)c, M, N, K, mt, (int)items);                                 \
    } while (0)
    switch (gemm_fp8_tile(M, N)) {
        case 4: G8(96, 128, 4, 1); break;
        case 0: G8(128, 128, 4, 1); break;
        case 1: G8(128, 128, 2, 2); break;
        case 2: G8(128, 256, 3, 1); break;
        default: G8(256, 256, 2, 1);
    }
#undef G8
    HIP_CHECK_LAUNCH();
    return 0;
}

// ---- MFMA fp8 GEMV v2 (decode path) ----------------------------------------
// The VALU dequant stream tops out at ~4.5-4.7 TB/s (~40 VALU ops per 16 W
// bytes). This path moves the multiply onto v_mfma_scale_f32_16x16x128_f8f6f4
// (identity E8M0 scales; per-row float scales in the epilogue — the tile
// GEMM's numerics): per 2 KiB of weights a lane issues 2 NT loads + 2 x
// loads + 1 MFMA instead of ~250 VALU ops.
//
// Occupancy is the real constraint (a first cut with 32-row waves and no
// K-split ran 1.1 TB/s: rows/32 waves x 8 outstanding loads = 40 KiB in
// flight vs the ~3.6 MB the HBM latency x bandwidth product demands), so:
//   * 16-row groups (16x16x128: B has 16 batch columns >= M)
//   * split-K on grid.y sized so blocks ~ 8192 (KS in {1..16} dividing K/128)
//   * partial f32 strips in a device-resident workspace; the LAST block of
//     each row-group (atomic counter, released/acquired with threadfences)
//     reduces the strips IN ORDER (deterministic fp sum) and applies
//     wscale[row]*xscale[m], the residual add, or the silu(g)*u pairing.
// x is pre-quantized to fp8 by quant_fp8_kernel (or its fused-rmsnorm
// variant below) in the same stream — two launches per GEMV total.
typedef __attribute__((ext_vector_type(4))) float f32x4_v;

// rmsnorm + per-row fp8 quant (the NORM prologue of the VALU gemv, moved
// into the quant step so the stream kernel sees finished fp8 activations)
__global__ __launch_bounds__(256) void quant_norm_fp8_kernel(
    const uint32_t* __restrict__ x,   // [T, K/2] bf16x2
    const uint32_t* __restrict__ wn,  // [K/2] rmsnorm weight
    uint32_t* __restrict__ q,         // [T, K/4]
    float* __restrict__ scales,       // [T]
    int T, int K, float eps) {
    const int row = blockIdx.x * 4 + threadIdx.x / WAVE;
    if (row >= T) return;
    const int lane = threadIdx.x & (WAVE - 1);
    const int k2 = K / 2;
    const uint32_t* xr = x + (size_t)row * k2;
    float ss = 0.0f, amax = 1e-8f;
    for (int i = lane * 4; i < k2; i += WAVE * 4) {
        uint4 w = *reinterpret_cast<const uint4*>(xr + i);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float lo = bf16_lo((&w.x)[j]), hi = bf16_hi((&w.x)[j]);
            ss = fmaf(lo, lo, ss);
            ss = fmaf(hi, hi, ss);
            const uint32_t g = wn[i + j];
            amax = fmaxf(amax, fabsf(lo * bf16_lo(g)));
            amax = fmaxf(amax, fabsf(hi * bf16_hi(g)));
        }
    }
    ss = wave_reduce_sum(ss);
    amax = wave_reduce_max(amax);
    const float rstd = rsqrtf(ss / (float)K + eps);
    amax *= rstd;
    const float inv = FP8_MAX / amax;
    if (lane == 0) scales[row] = amax / FP8_MAX;
    uint32_t* qr = q + (size_t)row * (K / 4);
    for (int i = lane * 4; i < k2; i += WAVE * 4) {
        uint4 w = *reinterpret_cast<const uint4*>(xr + i);
        uint2 o;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t g0 = wn[i + h * 2], g1 = wn[i + h * 2 + 1];
            unsigned packed = 0;
            packed = f32x2_to_fp8<false>(
                bf16_lo((&w.x)[h * 2]) * rstd * bf16_lo(g0) * inv,
                bf16_hi((&w.x)[h * 2]) * rstd * bf16_hi(g0) * inv, packed);
            packed = f32x2_to_fp8<true>(
                bf16_lo((&w.x)[h * 2 + 1]) * rstd * bf16_lo(g1) * inv,
                bf16_hi((&w.x)[h * 2 + 1]) * rstd * bf16_hi(g1) * inv, packed);
            (&o.x)[h] = packed;
        }
        *reinterpret_cast<uint2*>(qr + i / 2) = o;
    }
}

// Stream kernel: 256 threads; the FOUR waves split K (intra-block split-K:
// the f32 partial tiles meet in LDS — no cross-XCD fences, which made a
// grid-level split-K fixup 20x slower than the VALU path on this chip's
// per-XCD L2s). Wave w streams 16 W rows over k in [w*K/4, (w+1)*K/4) with
// a PF-deep register prefetch ring (PF=8 plain / 4 gateup: the in-flight
// byte product is what covers HBM latency — 16-row blocks x 4 waves x
// 256 B/lane ~ 40 MB chip-wide), x8 staged once to LDS.
template <bool GATEUP, bool ADDRES>
__global__ __launch_bounds__(256, 1) void gemv_fp8_mfma3_kernel(
    const uint32_t* __restrict__ x8,  // [M, K/4] fp8 (pre-quantized)
    const float* __restrict__ xsc,    // [M]
    const uint32_t* __restrict__ w8,  // [N, K/4] (gateup: [2I, K/4])
    const float* __restrict__ wscale, // [N] (gateup: [2I])
    uint32_t* __restrict__ out,       // [M, N] bf16 (gateup: [M, I])
    const uint32_t* __restrict__ res, // [M, N] residual (ADDRES)
    int M, int N, int K) {
    constexpr int PF = GATEUP ? 4 : 8;
    const int tid = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int wid = tid / WAVE;
    const int fr = lane & 15;   // A row / B,D col
    const int fs = lane >> 4;   // 32-byte k-slice; D rows fs*4..+3
    const int rows = GATEUP ? N / 2 : N;
    const int I = rows;
    const int row0 = blockIdx.x * 16;
    const int wrow = min(row0 + fr, rows - 1);

    // x8 image -> LDS (whole [M, K] fp8), plus the 4-wave reduction tiles
    extern __shared__ __attribute__((aligned(16))) char xls[];
    const int kw = K / 4;  // words per row
    for (int i = tid * 4; i < M * kw; i += 256 * 4)
        *reinterpret_cast<uint4*>(xls + i * 4) =
            *reinterpret_cast<const uint4*>(x8 + i);
    __syncthreads();

    const int klen = K / 4;              // bytes per wave
    const int k0 = wid * klen;
    const int nk = klen / 128;           // 128-B MFMA steps
    const char* wp = reinterpret_cast<const char*>(w8);
    const uint32_t* wr0 = reinterpret_cast<const uint32_t*>(
        wp + (size_t)wrow * K + k0) + fs * 8;
    const uint32_t* wr1 = reinterpret_cast<const uint32_t*>(
        wp + (size_t)(wrow + (GATEUP ? I : 0)) * K + k0) + fs * 8;
    const int xrow = fr < M ? fr : 0;
    const char* xr = xls + (size_t)xrow * K + k0 + fs * 32;

    f32x4_v acc0 = {}, acc1 = {};
    i32x8_f8 abuf[PF], ubuf[GATEUP ? PF : 1];
    auto load_a = [&](int p, int kb) {
        *reinterpret_cast<u32x4*>(&abuf[p]) = nt_load4f(wr0 + kb * 32);
        *(reinterpret_cast<u32x4*>(&abuf[p]) + 1) =
            nt_load4f(wr0 + kb * 32 + 4);
        if (GATEUP) {
            *reinterpret_cast<u32x4*>(&ubuf[p]) = nt_load4f(wr1 + kb * 32);
            *(reinterpret_cast<u32x4*>(&ubuf[p]) + 1) =
                nt_load4f(wr1 + kb * 32 + 4);
        }
    };
#pragma unroll
    for (int p = 0; p < PF; ++p) load_a(p, p);
    // x fragment double-buffered ONE step ahead (an inline ds_read feeding
    // its own MFMA serializes on lgkmcnt(0) every step)
    i32x8_f8 bcur;
    *reinterpret_cast<uint4*>(&bcur) = *reinterpret_cast<const uint4*>(xr);
    *(reinterpret_cast<uint4*>(&bcur) + 1) =
        *reinterpret_cast<const uint4*>(xr + 16);
    for (int kb0 = 0; kb0 < nk; kb0 += PF) {
        const bool more = kb0 + PF < nk;
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            const int kb = kb0 + p;
            i32x8_f8 bnext;
            if (kb + 1 < nk) {
                *reinterpret_cast<uint4*>(&bnext) =
                    *reinterpret_cast<const uint4*>(xr + (kb + 1) * 128);
                *(reinterpret_cast<uint4*>(&bnext) + 1) =
                    *reinterpret_cast<const uint4*>(xr + (kb + 1) * 128 + 16);
            }
            acc0 = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                abuf[p], bcur, acc0, 0, 0, 0, 0x7f, 0, 0x7f);
            if (GATEUP)
                acc1 = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                    ubuf[p], bcur, acc1, 0, 0, 0, 0x7f, 0, 0x7f);
            if (more) load_a(p, kb0 + PF + p);
            if (kb + 1 < nk) bcur = bnext;
        }
    }

    // intra-block reduction: [wave][plane][col fr][row fs*4+i] f32 in LDS
    __syncthreads();  // image reads done before the tiles overwrite it
    float* red = reinterpret_cast<float*>(xls);
    const int planes = GATEUP ? 2 : 1;
    {
        float* t = red + ((wid * planes) * 16 + fr) * 16 + fs * 4;
        *reinterpret_cast<f32x4_v*>(t) = acc0;
        if (GATEUP)
            *reinterpret_cast<f32x4_v*>(t + 16 * 16) = acc1;
    }
    __syncthreads();
    if (wid != 0 || fr >= M) return;
    const int m = fr;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = row0 + fs * 4 + i;
        if (row >= rows) continue;
        float sg = 0.0f, su = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            sg += red[((w * planes) * 16 + m) * 16 + fs * 4 + i];
            if (GATEUP)
                su += red[((w * planes + 1) * 16 + m) * 16 + fs * 4 + i];
        }
        float v;
        if (GATEUP) {
            const float gg = sg * wscale[row] * xsc[m];
            const float uu = su * wscale[row + I] * xsc[m];
            v = gg / (1.0f + __expf(-gg)) * uu;
        } else {
            v = sg * wscale[row] * xsc[m];
            if (ADDRES)
                v += bf16_to_f32(reinterpret_cast<const uint16_t*>(
                    res)[(size_t)m * rows + row]);
        }
        reinterpret_cast<uint16_t*>(out)[(size_t)m * rows + row] =
            f32_to_bf16(v);
    }
}

// device scratch for the pre-quantized x. Allocated ONCE on first use —
// callers must make a first (eager) call before any hipGraph capture; the
// engine's weight-quantization path does (ops.quant_fp8 wrapper).
static uint32_t* g_gemv8_x8 = nullptr;
static float* g_gemv8_xsc = nullptr;
#define GEMV8_MAX_M 16
#define GEMV8_MAX_K 32768

extern "C" int oa_fp8_gemv_scratch_init(void) {
    if (g_gemv8_x8) return 0;
    if (hipMalloc(&g_gemv8_x8, (size_t)GEMV8_MAX_M * GEMV8_MAX_K) != hipSuccess)
        return -1;
    if (hipMalloc(&g_gemv8_xsc, GEMV8_MAX_M * 4) != hipSuccess) return -1;
    return 0;
}

extern "C" int oa_gemv_fp8_mfma(void* stream, const void* x, const void* w8,
                                const void* wscale, void* out, const void* wn,
                                const void* res, int M, int N, int K,
                                float eps, int mode, int gateup) {
    const int rows = gateup ? N / 2 : N;
    if (K % 512 != 0 || (K / 512) % (gateup ? 4 : 8) != 0 ||
        M > GEMV8_MAX_M || K > GEMV8_MAX_K)
        return -100;
    const size_t img = (size_t)M * K;
    if (img > 128 * 1024) return -101;  // x image must fit LDS
    if (!g_gemv8_x8 && oa_fp8_gemv_scratch_init() != 0) return -102;
    hipStream_t s = (hipStream_t)stream;
    if (mode & 1) {
        hipLaunchKernelGGL(quant_norm_fp8_kernel, dim3(CEIL_DIV(M, 4)),
                           dim3(256), 0, s, (const uint32_t*)x,
                           (const uint32_t*)wn, g_gemv8_x8, g_gemv8_xsc, M, K,
                           eps);
    } else {
        quant_fp8<false>(s, x, g_gemv8_x8, g_gemv8_xsc, M, K);
    }
    const size_t shmem =
        img > (size_t)(gateup ? 2 : 1) * 4 * 16 * 16 * 4 * 4
            ? img
            : (size_t)(gateup ? 2 : 1) * 4 * 16 * 16 * 4 * 4;
    dim3 grid(CEIL_DIV(rows, 16)), block(256);
#define LAUNCH_MF3(GUV, RESV)                                                  \
    hipLaunchKernelGGL((gemv_fp8_mfma3_kernel<GUV, RESV>), grid, block, shmem, \
                       s, g_gemv8_x8, g_gemv8_xsc, (const uint32_t*)w8,        \
                       (const float*)wscale, (uint32_t*)out,                   \
                       (const uint32_t*)res, M, N, K)
    if (gateup) {
        LAUNCH_MF3(true, false);
    } else if (mode & 2) {
        LAUNCH_MF3(false, true);
    } else {
        LAUNCH_MF3(false, false);
    }
#undef LAUNCH_MF3
    HIP_CHECK_LAUNCH();
    return 0;
}
