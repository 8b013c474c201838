// Products of 2 to 128 rows with large weights: C[M, N] = x[M, K] W[N, K]^T in bf16, plain
// or gate-up with its activation. What bounds them is the weight stream, so everything
// serves to keep enough of it under way on every CU: both operands by direct transfers
// into a deep ring in LDS (no registers held by loads in flight), one or two blocks per CU,
// columns split where the strips alone would leave CUs idle, and weights read without being kept
// (nt) where they pass once: 5.9 TB/s, plain transfers of the same pieces reach 5.3. Us in
// graphs over 2 GB of weights, before (skinny.hip up to 32 rows, the library and the
// activation kernel above) / here: gate-up 2 x 14336 x 4096, M = 32 56.5 / 47.6, 47 55.7 /
// 49.5, 77 59.0 / 52.9; 4096 x 14336, M = 8 29.7 / 23.3, 47 40.0 / 27.1, 77 49.1 / 30.7, 128
// 75.4 / 33.5; 6144 x 4096, M = 8 17.4 / 13.2, 47 18.0 / 16.4, 77 22.7 / 18.0; 32000 x 4096,
// M = 32 57.8 / 48.5, 77 56.3 / 53.7; 8192 x 28672, M = 8 89.3 / 75.4, 47 140 / 81.0, 77
// 194 / 88.9. (The same over 0.5 GB reads up to a fifth better than inside a model.)
//
// Rows lie a few KiB apart, so blocks at the same columns read the same few memory channels, and
// all blocks start together. In bf16 each eight strips therefore start two steps further into
// their columns and go round. Us, together / apart: gate-up 2 x 14336 x 4096 in strips of 128, M =
// 8 46.6 / 36.6, 47 47.3 / 37.6 (6.2 TB/s), 77 49.9 / 41.6, 128 52.7 / 48.2; 32000 x 4096, 47 55.5 /
// 41.5, 77 57.4 / 43.8; in strips of 64, which had spread the starts some, M = 8 40.3 / 37.7 and 44.2
// / 40.8; 4096 x 14336 in seven splits, 47 32.0 / 30.4; 2 x 8192 x 2048, 8 15.3 / 13.3. Other steps
// between them were as good but one a strip (47.3); sixteen neighbours together too.
//
// Up to 64 rows a strip of 64 weight rows leaves LDS for two blocks a CU, whose rings keep
// more under way than one deep ring and start and end at different times; one strip more
// than fills the CUs no longer waits for a whole round either. Us, strips of 128 (or the
// other forms where those were faster) / 64: gate-up 2 x 14336 x 4096, M = 8 45.0 / 40.3, 32
// 45.4 / 42.7, 48 47.1 / 46.3; 32000 x 4096, M = 8 50.0 / 45.9, 24 51.1 / 44.7, 47 52.6 / 47.6;
// 2048 x 8192, M = 8 11.1 / 10.2, 47 14.1 / 12.1; 4096 x 4096, M = 24 11.8 / 10.4, 47 13.5 /
// 11.7; 3072 x 2048, M = 47 11.6 / 9.1. More rows are bound by what a CU reads of x, which
// narrow strips double: 32000 x 4096, M = 80 55.2 / 55.4, gate-up 2 x 14336 x 4096, M = 64
// 48.0 / 49.8, 80 49.3 / 54.1. There eight waves cover each other's waits better than four:
// gate-up 2 x 14336 x 4096, M = 64 51.1 / 49.7, 77 54.2 / 51.5; 4096 x 14336, 77 30.4 / 29.5, 128
// 34.1 / 32.4; fp8 28672 x 4096, 128 36.6 / 33.4. Sixteen are no faster, and tiles of 32 rows or
// narrow strips lose with eight (4096 x 4096 fp8, 8 8.6 / 9.1).
#include <type_traits>

#include "common.h"

typedef __attribute__((ext_vector_type(4))) float rgf4;
typedef __attribute__((ext_vector_type(8))) short rgs8;
typedef __attribute__((ext_vector_type(8))) int rgi8;

#define RG_MG(BM, RN) ((RN) > 64 && (BM) > 32 ? 2 : 1)   // groups of four waves of a block
#define RG_K 64                         // bf16 columns of a step: 128 bytes; fp8: 128

template <int V>
__device__ __forceinline__ void rg_wait() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(V) : "memory");
}

__device__ __forceinline__ float rg_gate(float g, float u, int act) {
    if (act == 2) {
        const float t = 0.7978845608028654f * fmaf(0.044715f * g * g, g, g);
        return 0.5f * g * (1.0f + tanhf(t)) * u;
    }
    return g / (1.0f + __expf(-g)) * u;
}

// A block of four waves, or of two such groups with half of the rows each, takes BM rows, a
// strip of RN = 128 or 64 weight rows (GU: half of them gate rows, half the up rows beside
// them) and one of `splits` runs of 64-column steps; a wave takes its rows by a quarter of the
// strip on v_mfma_f32_16x16x32_bf16, weights as
// the first operand, so that a lane ends with four neighbouring outputs of one row (GU: with
// gate and up of four outputs in its two fragments; in strips of 64 of two in its one, whose
// rows go gate, gate, up, up). Both operands come by 16-byte global_load_lds into a ring of
// STAGES steps: STAGES - 1 under way while one is in use, waits that leave the younger ones in flight (inline asm: hipcc's own waits
// drain builtin transfers before the first LDS read), one barrier per step, which says
// that the step has landed for every wave and that the one before is no longer read.
// 16-byte chunk c of row r lies at c ^ (r >> 1 & 7): the 16 rows of a fragment read
// touch every bank once. Weight rows past N and rows past M repeat the last one.
//
// F8: e4m3 rows on v_mfma_scale_f32_16x16x128_f8f6f4 with unit block scales (the tile
// product's arithmetic), a float32 scale per row of x and of w in the epilogue. us over 2 GB
// of weights, the tile product (fp8_moe.hip) / here: 28672 x 4096, M = 9 31.4 / 26.0, 77
// 37.5 / 31.1; 4096 x 14336, 9 66.3 / 14.9, 47 71.4 / 18.2, 128 78.9 / 26.5; 6144 x 4096, 47
// 26.9 / 13.2; 4096 x 4096, 77 28.6 / 14.9; 8192 x 28672, 77 140 / 46.8; 2048 x 2816, 33 20.0
// / 8.7.
template <int BM, int RN, int STAGES, bool GU, bool NT, bool F8>
__global__ __launch_bounds__(256 * RG_MG(BM, RN), RG_MG(BM, RN) == 2 || RN == 64 ? 2 : 1) void ring_gemm_kernel(
    const char* __restrict__ x, int64_t xs, const char* __restrict__ w,
    const float* __restrict__ xscale, const float* __restrict__ wscale,
    uint16_t* __restrict__ out, float* __restrict__ part, int M, int N, int K, int mtiles,
    int splits, int items, int act) {
    constexpr int MG = RG_MG(BM, RN), MT = BM / 16 / MG, NF = RN / 64;   // fragments of a wave
    constexpr int W = 4 * MG, TR = (RN + BM) / 8, LPS = (TR + W - 1) / W;    // transfers of a step, of a wave
    constexpr int STEP = (RN + BM) * 128;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int per = gridDim.x >> 3;
    const int item = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (item >= items) return;
    const int strip = item / (splits * mtiles), rest = item - strip * splits * mtiles;
    const int sp = rest / mtiles, m0 = (rest - sp * mtiles) * BM;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wid = wave & 3, mg = wave >> 2;
    const bool full = TR % W == 0 || wave < TR % W;  // the last waves have a transfer less
    const int64_t kb = F8 ? K : 2 * (int64_t)K;     // bytes of a weight row
    const int steps = (int)(kb / 128);
    const int s0 = (int)((int64_t)steps * sp / splits), s1 = (int)((int64_t)steps * (sp + 1) / splits);

    const int n = s1 - s0;
    // Strips start at steps of their own: rows lie some KiB apart, and blocks that all read the
    // same columns read the same few memory channels. Eight neighbours share a start. fp8 keeps
    // the order of its sums.
    const int turned = F8 ? 0 : (strip >> 3) * 2 % n;
    int ahead = n - turned;                          // steps to the last column

    // a transfer takes eight rows; this lane's row of it and its chunk
    const int lr = lane >> 3;
    const char* src[LPS];
    uint32_t dst[LPS];
#pragma unroll
    for (int p = 0; p < LPS; ++p) {
        const int tr = p * W + wave;
        const bool isw = tr < RN / 8;
        const int r = (isw ? tr : tr - RN / 8) * 8 + lr;
        const int chunk = (lane & 7) ^ (r >> 1 & 7);
        int64_t at;
        if (!isw) at = min(m0 + r, M - 1) * xs * (F8 ? 1 : 2);
        else if (GU && NF == 2) at = (min(strip * 64 + (r >> 5) * 16 + (r & 15), N - 1) + (r & 16 ? N : 0)) * kb;
        else if (GU) at = (min(strip * 32 + (r >> 2) * 2 + (r & 1), N - 1) + (r & 2 ? N : 0)) * kb;
        else at = min(strip * RN + r, N - 1) * kb;
        src[p] = (isw ? w : x) + at + (int64_t)(s0 + turned) * 128 + chunk * 16;
        dst[p] = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem + tr * 1024);
    }
    auto stage = [&](int buf) {
#pragma unroll
        for (int p = 0; p < LPS; ++p) {
            if (p == LPS - 1 && !full) break;
            if (NT && p * W + wave < RN / 8) lds_transfer16<true>(dst[p] + buf * STEP, src[p]);
            else lds_transfer16(dst[p] + buf * STEP, src[p]);
            src[p] += 128;
        }
        if (!F8 && --ahead == 0) {
#pragma unroll
            for (int p = 0; p < LPS; ++p) src[p] -= (int64_t)n * 128;
        }
    };
    auto wait = [&](auto count, int behind) {         // count: transfers of a step of this wave
        constexpr int C = decltype(count)::value;
        if (STAGES > 5 && behind >= 4) rg_wait<4 * C>();
        else if (STAGES > 4 && behind >= 3) rg_wait<3 * C>();
        else if (behind == 2) rg_wait<2 * C>();
        else if (behind == 1) rg_wait<C>();
        else rg_wait<0>();
    };
    rgf4 acc[NF][MT] = {};
#pragma unroll
    for (int t = 0; t < STAGES - 1; ++t)
        if (t < n) stage(t);
    int buf = 0;
    for (int t = 0; t < n; ++t) {
        const int behind = min(STAGES - 2, n - 1 - t);    // younger steps under way
        if (full) wait(std::integral_constant<int, LPS>(), behind);
        else wait(std::integral_constant<int, LPS - 1>(), behind);
        if (t + STAGES - 1 < n) stage(buf == 0 ? STAGES - 1 : buf - 1);
        const char* b = smem + buf * STEP;
        if constexpr (F8) {
            const int r = lane & 15, c = (lane >> 4) * 2;
            const int at = r * 128 + ((c ^ (r >> 1)) << 4), at2 = r * 128 + (((c + 1) ^ (r >> 1)) << 4);
            auto frag = [&](const char* rows) {
                union {
                    uint4 h[2];
                    rgi8 v;
                } f;
                f.h[0] = *reinterpret_cast<const uint4*>(rows + at);
                f.h[1] = *reinterpret_cast<const uint4*>(rows + at2);
                return f.v;
            };
            rgi8 wf[NF], xf[MT];
#pragma unroll
            for (int j = 0; j < NF; ++j) wf[j] = frag(b + (wid * NF + j) * 16 * 128);
#pragma unroll
            for (int m = 0; m < MT; ++m) xf[m] = frag(b + (RN + (mg * MT + m) * 16) * 128);
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int j = 0; j < NF; ++j)
                    acc[j][m] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                        wf[j], xf[m], acc[j][m], 0, 0, 0, 0x7f, 0, 0x7f);
        } else {
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                const int r = lane & 15, c = kk * 4 + (lane >> 4);
                const int at = r * 128 + ((c ^ (r >> 1)) << 4);         // rows step by 16: r >> 1 & 7 stays
                rgs8 wf[NF], xf[MT];
#pragma unroll
                for (int j = 0; j < NF; ++j)
                    wf[j] = *reinterpret_cast<const rgs8*>(b + (wid * NF + j) * 16 * 128 + at);
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    xf[m] = *reinterpret_cast<const rgs8*>(b + (RN + (mg * MT + m) * 16) * 128 + at);
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int j = 0; j < NF; ++j)
                        acc[j][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], xf[m], acc[j][m], 0, 0, 0);
            }
        }
        buf = buf + 1 == STAGES ? 0 : buf + 1;
    }
    // D: column (row of x) lane & 15, rows (weight rows) (lane >> 4) * 4 and up
    const int q = (lane >> 4) * 4;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int row = m0 + (mg * MT + m) * 16 + (lane & 15);
        if (row >= M) continue;
        if (GU && NF == 1) {
            const int col = strip * 32 + wid * 8 + q / 2;
            if (col >= N) continue;
            const rgf4 a = acc[0][m];
            if (part) {
                float* p = part + ((size_t)sp * M + row) * 2 * N + col;
                *reinterpret_cast<float2*>(p) = make_float2(a[0], a[1]);
                *reinterpret_cast<float2*>(p + N) = make_float2(a[2], a[3]);
            } else {
                *reinterpret_cast<uint32_t*>(out + (size_t)row * N + col) =
                    pack_bf16x2(rg_gate(a[0], a[2], act), rg_gate(a[1], a[3], act));
            }
        } else if (GU) {
            const int col = strip * 64 + wid * 16 + q;
            if (col >= N) continue;
            if (part) {
                float* p = part + ((size_t)sp * M + row) * 2 * N + col;
                *reinterpret_cast<rgf4*>(p) = acc[0][m];
                *reinterpret_cast<rgf4*>(p + N) = acc[NF - 1][m];
            } else {
                float o[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = rg_gate(acc[0][m][i], acc[NF - 1][m][i], act);
                *reinterpret_cast<uint2*>(out + (size_t)row * N + col) =
                    make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
            }
        } else {
#pragma unroll
            for (int j = 0; j < NF; ++j) {
                const int col = strip * RN + (wid * NF + j) * 16 + q;
                if (col >= N) continue;
                if (part) {
                    *reinterpret_cast<rgf4*>(part + ((size_t)sp * M + row) * N + col) = acc[j][m];
                    continue;
                }
                if (F8) {
                    const float sx = xscale[row];
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[j][m][i] = acc[j][m][i] * sx * wscale[col + i];
                }
                *reinterpret_cast<uint2*>(out + (size_t)row * N + col) =
                    make_uint2(pack_bf16x2(acc[j][m][0], acc[j][m][1]),
                               pack_bf16x2(acc[j][m][2], acc[j][m][3]));
            }
        }
    }
}

// parts [splits, M, N] (GU: [splits, M, 2 N]) added up in order
template <bool GU, bool F8>
__global__ __launch_bounds__(256) void ring_sum_kernel(const float* __restrict__ part,
                                                       const float* __restrict__ xscale,
                                                       const float* __restrict__ wscale,
                                                       uint16_t* __restrict__ out, int M, int N,
                                                       int splits, int act) {
    const int n4 = N / 4;
    const int c = blockIdx.x * blockDim.x + threadIdx.x, row = blockIdx.y;
    if (c >= n4) return;
    const size_t w = (GU ? 2 : 1) * (size_t)n4;
    const rgf4* p = reinterpret_cast<const rgf4*>(part) + row * w + c;
    rgf4 a = {}, u = {};
#pragma unroll 4
    for (int s = 0; s < splits; ++s) {
        a += p[(size_t)s * M * w];
        if (GU) u += p[(size_t)s * M * w + n4];
    }
    if (GU)
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = rg_gate(a[i], u[i], act);
    if (F8) {
        const float sx = xscale[row];
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = a[i] * sx * wscale[c * 4 + i];
    }
    reinterpret_cast<uint2*>(out)[(size_t)row * n4 + c] =
        make_uint2(pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]));
}

// out [M, N] = the sum of parts [splits, M, N], in order
extern "C" int oa_ring_sum(void* stream, const void* part, void* out, int M, int N, int splits) {
    if (M < 1 || M > 65535 || N < 4 || N % 4 != 0 || splits < 1 || !part || !out) return -100;
    if (((uintptr_t)part | (uintptr_t)out) % 16 != 0) return -102;
    const dim3 grid(CEIL_DIV(N / 4, 256), M);
    hipLaunchKernelGGL((ring_sum_kernel<false, false>), grid, dim3(256), 0, (hipStream_t)stream, (const float*)part,
                       (const float*)nullptr, (const float*)nullptr, (uint16_t*)out, M, N, splits, 0);
    HIP_CHECK_LAUNCH();
    return 0;
}

// out [M, N] = x [M, K] w [N, K]^T, x rows xs elements apart. act 1 (silu), 2 (tanh gelu):
// out = act(x w[:N]^T) * (x w[N:]^T), w [2 N, K]. bm: rows of a tile, 32, 64, 96 or 128;
// narrow: strips of 64 weight rows (bm 32 and 64).
// scratch: splits * M * N floats (act: twice that), unused at splits 1; out null: left
// there, not added up.
extern "C" int oa_ring_gemm(void* stream, const void* x, int64_t xs, const void* w, void* out,
                            void* scratch, int M, int N, int K, int bm, int narrow, int splits,
                            int act) {
    if (M < 1 || M > 65535 || N < 4 || N % 4 != 0 || K < RG_K || K % RG_K != 0) return -100;
    if (splits < 1 || splits > K / RG_K || (splits > 1 ? !scratch : !out)) return -101;
    if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out | (uintptr_t)scratch) % 16 != 0 || xs % 8 != 0)
        return -102;
    if (act < 0 || act > 2 || (bm != 32 && bm != 64 && bm != 96 && bm != 128) || (narrow && bm > 64)) return -104;
    const bool gateup = act != 0;
    const int mtiles = CEIL_DIV(M, bm);
    const int64_t items = (int64_t)CEIL_DIV(N, (narrow ? 64 : 128) / (gateup ? 2 : 1)) * mtiles * splits;
    if (items > (1 << 28)) return -103;
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid((unsigned)(CEIL_DIV(items, 8) * 8));
    float* part = splits > 1 ? (float*)scratch : nullptr;
#define RG(BMV, RNV, ST, G, NT)                                                                    \
    hipLaunchKernelGGL((ring_gemm_kernel<BMV, RNV, ST, G, NT, false>), grid,                        \
                       dim3(256 * RG_MG(BMV, RNV)),                                                 \
                       (ST) * ((RNV) + (BMV)) * 128, s, (const char*)x, xs, (const char*)w,         \
                       (const float*)nullptr, (const float*)nullptr, (uint16_t*)out, part, M, N, K, \
                       mtiles, splits, (int)items, act)
#define RGB(BMV, RNV, ST, NT)               \
    do {                                    \
        if (gateup) RG(BMV, RNV, ST, true, NT); \
        else RG(BMV, RNV, ST, false, NT);   \
    } while (0)
    // read without being kept: weights no other row tile reads, unless there are many rows
    // and few weights (us kept / not, 6144 x 4096, M = 8 14.3 / 13.2, 77 18.2 / 20.2; 2 x 8192
    // x 2048, 47 18.5 / 16.4; 8192 x 28672, 77 98.9 / 88.6)
    const bool nt = mtiles == 1 && (bm == 32 || (int64_t)N * K * (gateup ? 2 : 1) >= 32000000);
    if (narrow && bm == 32) RGB(32, 64, 6, true);
    else if (narrow && nt) RGB(64, 64, 4, true);
    else if (narrow) RGB(64, 64, 4, false);
    else if (bm == 32) RGB(32, 128, 6, true);
    else if (bm == 64 && nt) RGB(64, 128, 5, true);
    else if (bm == 64) RGB(64, 128, 5, false);
    else if (bm == 96 && nt) RGB(96, 128, 5, true);
    else if (bm == 96) RGB(96, 128, 5, false);
    else if (nt) RGB(128, 128, 4, true);
    else RGB(128, 128, 4, false);
#undef RGB
#undef RG
    if (splits > 1 && out) {
        const dim3 g(CEIL_DIV(N / 4, 256), M);
        if (gateup)
            hipLaunchKernelGGL((ring_sum_kernel<true, false>), g, dim3(256), 0, s, part,
                               (const float*)nullptr, (const float*)nullptr, (uint16_t*)out, M, N,
                               splits, act);
        else
            hipLaunchKernelGGL((ring_sum_kernel<false, false>), g, dim3(256), 0, s, part,
                               (const float*)nullptr, (const float*)nullptr, (uint16_t*)out, M, N,
                               splits, 0);
    }
    HIP_CHECK_LAUNCH();
    return 0;
}

// out [M, N] = (x8 [M, K] w8 [N, K]^T) * xscale[m] * wscale[n]; bm as above (several row
// tiles: 128), scratch as above
extern "C" int oa_ring_gemm_fp8(void* stream, const void* x8, const void* xscale, const void* w8,
                                const void* wscale, void* out, void* scratch, int M, int N, int K,
                                int bm, int splits) {
    if (M < 1 || M > 65535 || N < 4 || N % 4 != 0 || K < 128 || K % 128 != 0) return -100;
    if (splits < 1 || splits > K / 128 || (splits > 1 && !scratch)) return -101;
    if (((uintptr_t)x8 | (uintptr_t)w8 | (uintptr_t)out | (uintptr_t)scratch) % 16 != 0) return -102;
    if ((bm != 32 && bm != 64 && bm != 96 && bm != 128) || (M > bm && bm != 128)) return -104;
    const int mtiles = CEIL_DIV(M, bm);
    const int64_t items = (int64_t)CEIL_DIV(N, 128) * mtiles * splits;
    if (items > (1 << 28)) return -103;
    hipStream_t s = (hipStream_t)stream;
    float* part = splits > 1 ? (float*)scratch : nullptr;
#define RG8(BMV, ST, NT)                                                                           \
    hipLaunchKernelGGL((ring_gemm_kernel<BMV, 128, ST, false, NT, true>),                               \
                       dim3((unsigned)(CEIL_DIV(items, 8) * 8)), dim3(256 * RG_MG(BMV, 128)),      \
                       (ST) * (128 + (BMV)) * 128, s, (const char*)x8, (int64_t)K, (const char*)w8, \
                       (const float*)xscale, (const float*)wscale, (uint16_t*)out, part, M, N, K,  \
                       mtiles, splits, (int)items, 0)
    if (bm == 32) RG8(32, 6, true);
    else if (bm == 64) RG8(64, 5, true);
    else if (bm == 96) RG8(96, 5, true);
    else if (mtiles == 1) RG8(128, 4, true);
    else RG8(128, 4, false);
#undef RG8
    if (splits > 1)
        hipLaunchKernelGGL((ring_sum_kernel<false, true>), dim3(CEIL_DIV(N / 4, 256), M), dim3(256), 0, s,
                           part, (const float*)xscale, (const float*)wscale, (uint16_t*)out, M, N,
                           splits, 0);
    HIP_CHECK_LAUNCH();
    return 0;
}
