// Products of a few activation rows with a streamed weight:
//   out[M, N] = x[M, K] @ w[N, K]^T,  or  act(x @ gate^T) * (x @ up^T),  bf16
// for M up to 32 (batched decode). A pass is bound by the weight's bytes, and what
// keeps it from them is the activations: a block that stages them in LDS first has
// nothing in flight meanwhile (3.7 TB/s on 28672 x 4096 with 8 rows).
//
// Both forms load weight rows from memory straight into the A fragments of
// v_mfma_f32_16x16x32_bf16, several steps of 32 columns ahead (16 rows x 64 bytes
// per load read 6.0 TB/s with plain loads, 5.2 with non-temporal ones) and cut K
// between the waves of a block, whose partial sums meet in LDS.
//   strips:     a block takes one strip of 16 weight rows (a gate strip and the up
//               strip beside it) and reads its activation fragments from the L2 as
//               it goes. Every strip reads all of x: the form for few rows of x or
//               few strips.
//   persistent: a block keeps its activation fragments in registers and goes over
//               many strips. K = 4096 (16 waves x 8 steps).
// us, weights of 1 GiB in turn, strips / persistent / the library / staged in LDS
// (M up to 8): 28672 x 4096 gate-up, M = 3 46.4 / 40.6 / 61 / 58, 8 48.5 / 41.3 / 62 /
// 60, 16 54 / 43.6 / 63 / -; 6144 x 4096, M = 8 14.6 / 12.8 / 15.2 / 16.8; 4096 x
// 4096, M = 8 9.0 / 9.7 / 15.6 / 10.5, 16 10.6 / 11.6 / 15.5 / -; 32000 x 4096, M = 8
// 54 / 46 / 60 / 62, 32 101 / 53.6 / 65 / -; 16384 x 2048 gate-up, M = 8 14.2 / - /
// 18.7 / 18.9; 2048 x 2816, M = 13 7.5 / - / 11.3 / -; 4096 x 14336, M = 3 22.0 / - /
// 26.5 / -, 16 35 / - / 27 / -.
#include "skinny_strip.h"

template <int MF, bool GU, int WV, int D>
__global__ __launch_bounds__(WV * 64) void skinny_strip_kernel(
    const uint16_t* __restrict__ x, int64_t xs, const uint16_t* __restrict__ w,
    uint16_t* __restrict__ out, int M, int N, int K, int act) {
    __shared__ __attribute__((aligned(16))) SkinnyRed<MF, GU, WV> red;
    skinny_strip<MF, GU, WV, D>(x, xs, w, out, M, N, K, act, blockIdx.x, red);
}

// Two products of equal sizes in one launch (strips, up to 16 rows): one after the other they are a launch of
// 5 us each, whose strips of short rows end before the chip is full. us, 3 rows of 256 columns against 4096
// weight rows twice, traced one by one: 10.0 / 5.5.
template <int WV>
__global__ __launch_bounds__(WV * 64) void skinny_pair_kernel(
    const uint16_t* __restrict__ x0, const uint16_t* __restrict__ x1, int64_t xs, const uint16_t* __restrict__ w0,
    const uint16_t* __restrict__ w1, uint16_t* __restrict__ out0, uint16_t* __restrict__ out1, int M, int N, int K,
    int units) {
    __shared__ __attribute__((aligned(16))) SkinnyRed<1, false, WV> red;
    const bool second = (int)blockIdx.x >= units;
    skinny_strip<1, false, WV, 8>(second ? x1 : x0, xs, second ? w1 : w0, second ? out1 : out0, M, N, K, 0,
                                  second ? blockIdx.x - units : blockIdx.x, red);
}

// Strips go gate, up, gate, up; a register of the ring is refilled with the next
// strip's columns as soon as it is used, so a wave always has SW loads of 1 KiB in
// flight, across the barrier of the partial sums too (two LDS buffers, one barrier
// per output strip). After the last strip the ring is refilled with itself.
template <int MF, bool GU, int WV, int SW>
__global__ __launch_bounds__(WV * 64) void skinny_persistent_kernel(
    const uint16_t* __restrict__ x, int64_t xs, const uint16_t* __restrict__ w,
    uint16_t* __restrict__ out, int M, int N, int units, int act) {
    constexpr int RT = GU ? 2 : 1, K = WV * SW * 32;
    __shared__ __attribute__((aligned(16))) float red[2][WV][RT][MF][16][20];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int r = lane & 15, q = lane >> 4;
    const int c0 = wid * SW * 32 + q * 8;
    auto strip = [&](int u, int t) { return w + (size_t)(min(u * 16 + r, N - 1) + (t ? N : 0)) * K + c0; };
    int u = blockIdx.x, t = 0, buf = 0;
    const uint16_t* p = strip(u, 0);
    sk_u4 wb[SW];
#pragma unroll
    for (int s = 0; s < SW; ++s) wb[s] = *reinterpret_cast<const sk_u4*>(p + s * 32);
    sk_b8 xb[SW][MF];
#pragma unroll
    for (int f = 0; f < MF; ++f) {
        const uint16_t* xp = x + (size_t)min(f * 16 + r, M - 1) * xs + c0;
#pragma unroll
        for (int s = 0; s < SW; ++s) xb[s][f] = *reinterpret_cast<const sk_b8*>(xp + s * 32);
    }
    for (;;) {
        const int nu = GU && !t ? u : u + (int)gridDim.x, nt = GU && !t ? 1 : 0;
        const bool last = nu >= units;
        p = last ? p : strip(nu, nt);
        sk_f4 acc[MF];
#pragma unroll
        for (int f = 0; f < MF; ++f) acc[f] = sk_f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < SW; ++s) {
#pragma unroll
            for (int f = 0; f < MF; ++f)
                acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(sk_b8, wb[s]), xb[s][f],
                                                                 acc[f], 0, 0, 0);
            wb[s] = *reinterpret_cast<const sk_u4*>(p + s * 32);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int f = 0; f < MF; ++f) *reinterpret_cast<sk_f4*>(&red[buf][wid][t][f][r][q * 4]) = acc[f];
        if (!GU || t) {
            __syncthreads();
            for (int i = tid; i < MF * 256; i += WV * 64) {
                const int c = i & 15, m = (i >> 4) & 15, f = i >> 8;
                const int row = f * 16 + m, n = u * 16 + c;
                if (row >= M || n >= N) continue;
                float a = 0.0f, b = 0.0f;
#pragma unroll
                for (int v = 0; v < WV; ++v) {
                    a += red[buf][v][0][f][m][c];
                    if (GU) b += red[buf][v][RT - 1][f][m][c];
                }
                out[(size_t)row * N + n] = f32_to_bf16(GU ? sk_gate(a, act) * b : a);
            }
            buf ^= 1;
        }
        if (last) break;
        u = nu;
        t = nt;
    }
}

// gateup: w [2N, K], gate rows first; act 0 silu, 1 gelu in its tanh form.
// form 1: strips, 2: persistent (K = 4096; gate-up for M <= 16 only). xs: elements between rows of x.
extern "C" int oa_skinny(void* stream, const void* x, int64_t xs, const void* w, void* out, int M,
                         int N, int K, int gateup, int act, int form) {
    if (M < 1 || M > 32 || N < 1 || K < 32 || K % 32 != 0 || xs % 8 != 0 || xs < K) return -100;
    hipStream_t st = (hipStream_t)stream;
    const int units = CEIL_DIV(N, 16);
    if (form == 2) {
        if (K != 4096) return -101;
        // one block per CU, every block the same number of strips
        const dim3 grid(CEIL_DIV(units, CEIL_DIV(units, 256)));
#define SKP(MF, GU)                                                                             \
    hipLaunchKernelGGL((skinny_persistent_kernel<MF, GU, 16, 8>), grid, dim3(1024), 0, st,      \
                       (const uint16_t*)x, xs, (const uint16_t*)w, (uint16_t*)out, M, N, units, act)
        if (M <= 16) {
            if (gateup) SKP(1, true);
            else SKP(1, false);
        } else {
            if (gateup) return -103;   // gate and up partial sums of 32 rows fill the LDS
            SKP(2, false);
        }
#undef SKP
    } else if (form == 1) {
#define SKS(MF, GU, WV, D)                                                                      \
    hipLaunchKernelGGL((skinny_strip_kernel<MF, GU, WV, D>), dim3(units), dim3((WV) * 64), 0, st, \
                       (const uint16_t*)x, xs, (const uint16_t*)w, (uint16_t*)out, M, N, K, act)
        // four waves where K is short, and where few strips are long ones (4096 x
        // 14336, M = 3: 22.0 us with four waves, 25.3 with eight)
        if (gateup) {
            if (M > 16) SKS(2, true, 8, 4);
            else if (K <= 2048) SKS(1, true, 4, 8);
            else SKS(1, true, 8, 8);
        } else {
            if (M > 16) SKS(2, false, 8, 4);
            else if (K >= 2 * N) SKS(1, false, 4, 8);
            else SKS(1, false, 8, 8);
        }
#undef SKS
    } else {
        return -102;
    }
    HIP_CHECK_LAUNCH();
    return 0;
}

// out0 = x0 w0^T and out1 = x1 w1^T, [M, N] of up to 16 rows xs elements apart, the strips of oa_skinny
extern "C" int oa_skinny_pair(void* stream, const void* x0, const void* x1, int64_t xs, const void* w0, const void* w1,
                              void* out0, void* out1, int M, int N, int K) {
    if (M < 1 || M > 16 || N < 1 || K < 32 || K % 32 != 0 || xs % 8 != 0 || xs < K) return -100;
    if (!x0 || !x1 || !w0 || !w1 || !out0 || !out1) return -101;
    if (((uintptr_t)x0 | (uintptr_t)x1 | (uintptr_t)w0 | (uintptr_t)w1) % 16 != 0) return -102;
    const int units = CEIL_DIV(N, 16);
#define SKT(WV)                                                                                                 \
    hipLaunchKernelGGL((skinny_pair_kernel<WV>), dim3(2 * units), dim3((WV) * 64), 0, (hipStream_t)stream,      \
                       (const uint16_t*)x0, (const uint16_t*)x1, xs, (const uint16_t*)w0, (const uint16_t*)w1,  \
                       (uint16_t*)out0, (uint16_t*)out1, M, N, K, units)
    if (K >= 2 * N) SKT(4);                          // as oa_skinny
    else SKT(8);
#undef SKT
    HIP_CHECK_LAUNCH();
    return 0;
}
