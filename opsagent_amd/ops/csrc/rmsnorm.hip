// RMSNorm kernels for MI355X (gfx950) — memory-bound, HBM-roofline targets.
//
// One 256-thread block per row, 16-byte loads (scalar bf16 2.35 TB/s, vectorized
// 4.89 TB/s), f32 accumulation, wave + LDS block reduce; the residual-add variant
// writes both the normed output and the new residual stream in one pass.

#include "common.h"

// One block per row, D a multiple of 8 up to 8192; a thread takes 8 columns of each 2048.
// ADD: x + residual, which is written back. EMBED: x's row is the table's for the row's
// token, and becomes the residual: one launch for the gather and the norm of a step's
// first layer, which the library walks token by token up to 16 of them (us, gather and
// norm in a step of 8 rows of 4096: 7.7 + 4.4, of 16 of 2048 10.8 + 4.8; a step of 13
// tokens through experts 590 -> 580, of 8 sequences 505 -> 502, of 47 885 -> 866). An id
// outside the table, which the engine refuses before, gets a row of NaN.
// SCALES (float): out is the normed row as quant_fp8 (fp8_moe.hip) would leave it, of the same bf16 values: 8-bit
// numbers [rows, D] and a scale a row. One launch, 8 KB a row of 4096 out and in again less: us of a
// layer's norm and quantization in a run of products, 700 rows of 4096 11.3 -> 6.6, 20 rows 9.3 -> 4.9.
enum { RN_PLAIN, RN_ADD, RN_EMBED };
template <int MODE, typename ID, typename... SCALES>
__global__ __launch_bounds__(256) void rmsnorm_kernel(
    const uint4* __restrict__ x,      // [rows, D / 8] packed bf16
    uint4* __restrict__ residual,     // [rows, D / 8] in/out (ADD), out (EMBED)
    const uint4* __restrict__ w, uint4* __restrict__ out, const ID* __restrict__ ids, int64_t vocab,
    int D8, float inv_d, float eps, SCALES*... scales) {
    constexpr bool QUANT = sizeof...(SCALES) > 0;
    __shared__ float red[16];
    const int64_t row = blockIdx.x;
    int64_t from = row;
    bool known = true;                               // the same for the block
    if (MODE == RN_EMBED) {
        from = ids[row];
        known = from >= 0 && from < vocab;
        if (!known) from = 0;                        // loads behind a branch wait one by one
    }
    const uint4* xrow = x + from * D8;
    float v[4][8], sumsq = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int c = k * 256 + threadIdx.x;
        if (c >= D8) break;
        const uint32_t nan = 0x7fc07fc0u;
        uint4 xv = xrow[c];
        if (MODE == RN_EMBED && !known) xv = make_uint4(nan, nan, nan, nan);
        uint4 r;
        if (MODE == RN_ADD) r = residual[row * D8 + c];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float lo = bf16_lo((&xv.x)[j]), hi = bf16_hi((&xv.x)[j]);
            if (MODE == RN_ADD) {
                lo += bf16_lo((&r.x)[j]);
                hi += bf16_hi((&r.x)[j]);
                (&r.x)[j] = pack_bf16x2(lo, hi);
            }
            v[k][2 * j] = lo;
            v[k][2 * j + 1] = hi;
            sumsq += lo * lo + hi * hi;
        }
        if (MODE != RN_PLAIN) residual[row * D8 + c] = MODE == RN_ADD ? r : xv;
    }
    const float scale = rsqrtf(block_reduce_sum<16>(sumsq, red) * inv_d + eps);
    float amax = 1e-8f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int c = k * 256 + threadIdx.x;
        if (c >= D8) break;
        const uint4 g = w[c];
        uint4 o;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            (&o.x)[j] = pack_bf16x2(v[k][2 * j] * scale * bf16_lo((&g.x)[j]),
                                    v[k][2 * j + 1] * scale * bf16_hi((&g.x)[j]));
            if (QUANT) {
                v[k][2 * j] = bf16_lo((&o.x)[j]);
                v[k][2 * j + 1] = bf16_hi((&o.x)[j]);
                amax = fmaxf(amax, fmaxf(fabsf(v[k][2 * j]), fabsf(v[k][2 * j + 1])));
            }
        }
        if (!QUANT) out[row * D8 + c] = o;
    }
    if (!QUANT) return;
    __shared__ float most[4];
    amax = wave_reduce_max(amax);
    if ((threadIdx.x & (WAVE - 1)) == 0) most[threadIdx.x / WAVE] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(most[0], most[1]), fmaxf(most[2], most[3]));
    const float inv = 448.0f / amax;                 // the largest e4m3 number
    if (threadIdx.x == 0) ((scales[row] = amax / 448.0f), ...);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int c = k * 256 + threadIdx.x;
        if (c >= D8) break;
        uint2 o;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float* f = v[k] + 4 * h;
            const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[0] * inv, f[1] * inv, 0, false);
            (&o.x)[h] = __builtin_amdgcn_cvt_pk_fp8_f32(f[2] * inv, f[3] * inv, lo, true);
        }
        reinterpret_cast<uint2*>(out)[row * D8 + c] = o;
    }
}

template <int MODE, typename ID = int64_t>
static int launch_rmsnorm(void* stream, const void* x, void* residual, const void* w, void* out,
                          const void* ids, int64_t vocab, int rows, int dim, float eps) {
    if (dim % 8 != 0 || dim > 8192) return -100;
    hipLaunchKernelGGL((rmsnorm_kernel<MODE, ID>), dim3(rows), dim3(256), 0, (hipStream_t)stream,
                       (const uint4*)x, (uint4*)residual, (const uint4*)w, (uint4*)out,
                       (const ID*)ids, vocab, dim / 8, 1.0f / dim, eps);
    HIP_CHECK_LAUNCH();
    return 0;
}

extern "C" int oa_rmsnorm(void* stream, const void* x, const void* w, void* out,
                          int rows, int dim, float eps) {
    return launch_rmsnorm<RN_PLAIN>(stream, x, nullptr, w, out, nullptr, 0, rows, dim, eps);
}

extern "C" int oa_fused_add_rmsnorm(void* stream, const void* x, void* residual,
                                    const void* w, void* out, int rows, int dim,
                                    float eps) {
    return launch_rmsnorm<RN_ADD>(stream, x, residual, w, out, nullptr, 0, rows, dim, eps);
}

// x + residual, written back, and its norm in 8 bits: q [rows, dim], scales [rows]
extern "C" int oa_fused_add_rmsnorm_fp8(void* stream, const void* x, void* residual, const void* w, void* q,
                                        void* scales, int rows, int dim, float eps) {
    if (rows < 1 || dim % 8 != 0 || dim > 8192) return -100;
    if (((uintptr_t)x | (uintptr_t)residual | (uintptr_t)w) % 16 != 0 || (uintptr_t)q % 8 != 0) return -101;
    hipLaunchKernelGGL((rmsnorm_kernel<RN_ADD, int64_t, float>), dim3(rows), dim3(256), 0, (hipStream_t)stream,
                       (const uint4*)x, (uint4*)residual, (const uint4*)w, (uint4*)q, (const int64_t*)nullptr,
                       (int64_t)0, dim / 8, 1.0f / dim, eps, (float*)scales);
    HIP_CHECK_LAUNCH();
    return 0;
}

// ids: int64 (wide) or int32 token of every row of the table [vocab, dim]
extern "C" int oa_embed_rmsnorm(void* stream, const void* table, const void* ids, int wide,
                                int64_t vocab, const void* w, void* residual, void* out, int rows,
                                int dim, float eps) {
    if (rows < 1) return 0;
    if (vocab < 1) return -102;
    if (((uintptr_t)table | (uintptr_t)residual | (uintptr_t)w | (uintptr_t)out) % 16 != 0) return -101;
    if (wide) return launch_rmsnorm<RN_EMBED, int64_t>(stream, table, residual, w, out, ids, vocab, rows, dim, eps);
    return launch_rmsnorm<RN_EMBED, int>(stream, table, residual, w, out, ids, vocab, rows, dim, eps);
}

// The same behind a product whose columns are split: x is the sum of `parts` float32 planes
// [parts, rows, D], added in order and rounded to bf16 as the product by itself would be. One
// launch less per product, us of the sum and the norm / of this, 64 rows of 4096 in 8
// planes: 9.6 / 5.2. What bounds it is the launch and one round of loads: a thread takes
// four columns of all planes.
__global__ __launch_bounds__(1024) void rmsnorm_parts_kernel(
    const float* __restrict__ x, int parts, int64_t plane, uint16_t* __restrict__ residual,
    const uint16_t* __restrict__ w, uint16_t* __restrict__ out, int D, float inv_d, float eps) {
    __shared__ float red[16];
    const float* xrow = x + (int64_t)blockIdx.x * D;
    uint16_t* rrow = residual + (int64_t)blockIdx.x * D;
    float v[2][4];
    float sumsq = 0.0f;
#pragma unroll
    for (int k = 0; k < 2; ++k) {                    // D <= 8192
        const int c = (k * 1024 + threadIdx.x) * 4;
        if (c >= D) break;
        const uint2 r = *reinterpret_cast<const uint2*>(rrow + c);
        float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll 8
        for (int s = 0; s < parts; ++s) {
            const float4 y = *reinterpret_cast<const float4*>(xrow + s * plane + c);
            a.x += y.x;
            a.y += y.y;
            a.z += y.z;
            a.w += y.w;
        }
        const uint32_t lo = pack_bf16x2(a.x, a.y), hi = pack_bf16x2(a.z, a.w);
        v[k][0] = bf16_lo(lo) + bf16_lo(r.x);
        v[k][1] = bf16_hi(lo) + bf16_hi(r.x);
        v[k][2] = bf16_lo(hi) + bf16_lo(r.y);
        v[k][3] = bf16_hi(hi) + bf16_hi(r.y);
#pragma unroll
        for (int j = 0; j < 4; ++j) sumsq += v[k][j] * v[k][j];
        *reinterpret_cast<uint2*>(rrow + c) =
            make_uint2(pack_bf16x2(v[k][0], v[k][1]), pack_bf16x2(v[k][2], v[k][3]));
    }
    const float scale = rsqrtf(block_reduce_sum<16>(sumsq, red) * inv_d + eps);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int c = (k * 1024 + threadIdx.x) * 4;
        if (c >= D) break;
        const uint2 g = *reinterpret_cast<const uint2*>(w + c);
        *reinterpret_cast<uint2*>(out + (int64_t)blockIdx.x * D + c) =
            make_uint2(pack_bf16x2(v[k][0] * scale * bf16_lo(g.x), v[k][1] * scale * bf16_hi(g.x)),
                       pack_bf16x2(v[k][2] * scale * bf16_lo(g.y), v[k][3] * scale * bf16_hi(g.y)));
    }
}

extern "C" int oa_add_rmsnorm_parts(void* stream, const void* x, int parts, void* residual,
                                    const void* w, void* out, int rows, int dim, float eps) {
    if (dim % 8 != 0 || dim > 8192 || parts < 1 || rows < 1) return -100;
    if (((uintptr_t)x | (uintptr_t)residual | (uintptr_t)w | (uintptr_t)out) % 16 != 0) return -101;
    const int threads = dim >= 4096 ? 1024 : CEIL_DIV(dim / 4, WAVE) * WAVE;
    hipLaunchKernelGGL(rmsnorm_parts_kernel, dim3(rows), dim3(threads), 0, (hipStream_t)stream,
                       (const float*)x, parts, (int64_t)rows * dim, (uint16_t*)residual,
                       (const uint16_t*)w, (uint16_t*)out, dim, 1.0f / dim, eps);
    HIP_CHECK_LAUNCH();
    return 0;
}

// The same behind routed experts: x is the sum of a token's `top` rows of y [rows * top, D],
// bf16, and its row of `more` if there is one, in that order in float32, rounded to bf16 as
// the sum by itself would be. One launch and one pass less: a decode step of 13 tokens over 4
// layers of 64 experts 599 -> 586 us, a prompt of 512 1427 -> 1418.
// PARTS: `more` is still the n float32 planes [rows, 8 * D8] of its product, added up and rounded as the
// product alone would be: a prompt of 512 over those layers 1313 -> 1305.
template <bool PARTS>
__global__ __launch_bounds__(1024) void rmsnorm_pairs_kernel(
    const uint4* __restrict__ y, int top, const uint4* __restrict__ more, int n,
    uint4* __restrict__ residual, const uint4* __restrict__ w, uint4* __restrict__ out, int D8,
    float inv_d, float eps) {
    __shared__ float red[16];
    const int c = threadIdx.x;                       // eight columns
    const int64_t at = (int64_t)blockIdx.x * D8 + c;
    float v[8], sumsq = 0.0f;
    uint4 g;
    if (c < D8) {
        const uint4 r = residual[at];
        g = w[c];
        uint4 m = make_uint4(0, 0, 0, 0);
        if (PARTS) {
            float p[8] = {};
#pragma unroll 4
            for (int k = 0; k < n; ++k)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const float4 u = reinterpret_cast<const float4*>(more)[((int64_t)k * gridDim.x * D8 + at) * 2 + h];
                    p[4 * h] += u.x;
                    p[4 * h + 1] += u.y;
                    p[4 * h + 2] += u.z;
                    p[4 * h + 3] += u.w;
                }
#pragma unroll
            for (int j = 0; j < 4; ++j) (&m.x)[j] = pack_bf16x2(p[2 * j], p[2 * j + 1]);
        } else if (more) {
            m = more[at];
        }
        const uint4* row = y + (int64_t)blockIdx.x * top * D8 + c;
        float a[8] = {};
#pragma unroll 8
        for (int k = 0; k < top; ++k) {
            const uint4 u = row[(int64_t)k * D8];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                a[2 * j] += bf16_lo((&u.x)[j]);
                a[2 * j + 1] += bf16_hi((&u.x)[j]);
            }
        }
        uint4 o;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (more) {
                a[2 * j] += bf16_lo((&m.x)[j]);
                a[2 * j + 1] += bf16_hi((&m.x)[j]);
            }
            const uint32_t x = pack_bf16x2(a[2 * j], a[2 * j + 1]);
            v[2 * j] = bf16_lo(x) + bf16_lo((&r.x)[j]);
            v[2 * j + 1] = bf16_hi(x) + bf16_hi((&r.x)[j]);
            sumsq += v[2 * j] * v[2 * j] + v[2 * j + 1] * v[2 * j + 1];
            (&o.x)[j] = pack_bf16x2(v[2 * j], v[2 * j + 1]);
        }
        residual[at] = o;
    }
    const float scale = rsqrtf(block_reduce_sum<16>(sumsq, red) * inv_d + eps);
    if (c >= D8) return;
    uint4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        (&o.x)[j] = pack_bf16x2(v[2 * j] * scale * bf16_lo((&g.x)[j]),
                                v[2 * j + 1] * scale * bf16_hi((&g.x)[j]));
    out[at] = o;
}

extern "C" int oa_add_rmsnorm_pairs(void* stream, const void* y, int top, const void* more,
                                    void* residual, const void* w, void* out, int rows, int dim,
                                    float eps) {
    if (dim % 8 != 0 || dim > 8192 || top < 1 || rows < 1) return -100;
    if (((uintptr_t)y | (uintptr_t)more | (uintptr_t)residual | (uintptr_t)w | (uintptr_t)out) % 16 != 0)
        return -101;
    hipLaunchKernelGGL((rmsnorm_pairs_kernel<false>), dim3(rows), dim3(CEIL_DIV(dim / 8, WAVE) * WAVE), 0,
                       (hipStream_t)stream, (const uint4*)y, top, (const uint4*)more, 0,
                       (uint4*)residual, (const uint4*)w, (uint4*)out, dim / 8, 1.0f / dim, eps);
    HIP_CHECK_LAUNCH();
    return 0;
}

// more: n float32 planes [rows, dim]
extern "C" int oa_add_rmsnorm_pairs_parts(void* stream, const void* y, int top, const void* more, int n,
                                          void* residual, const void* w, void* out, int rows, int dim, float eps) {
    if (dim % 8 != 0 || dim > 8192 || top < 1 || rows < 1 || n < 1 || !more) return -100;
    if (((uintptr_t)y | (uintptr_t)more | (uintptr_t)residual | (uintptr_t)w | (uintptr_t)out) % 16 != 0)
        return -101;
    hipLaunchKernelGGL((rmsnorm_pairs_kernel<true>), dim3(rows), dim3(CEIL_DIV(dim / 8, WAVE) * WAVE), 0,
                       (hipStream_t)stream, (const uint4*)y, top, (const uint4*)more, n,
                       (uint4*)residual, (const uint4*)w, (uint4*)out, dim / 8, 1.0f / dim, eps);
    HIP_CHECK_LAUNCH();
    return 0;
}
