// The strip product of a few activation rows (skinny.hip, where the figures are), as a part that
// other launches have beside what they do.
#pragma once

#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 sk_b8;
typedef __attribute__((ext_vector_type(4))) float sk_f4;
typedef __attribute__((ext_vector_type(4))) unsigned int sk_u4;

__device__ __forceinline__ float sk_gate(float g, int act) {
    if (act == 1) {
        const float t = tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g));
        return 0.5f * g * (1.0f + t);
    }
    return g / (1.0f + __expf(-g));
}

// partial sums of a block's waves
template <int MF, bool GU, int WV>
struct SkinnyRed {
    float at[WV][GU ? 2 : 1][MF][16][20];
};

// One strip by a block of WV waves
template <int MF, bool GU, int WV, int D>
__device__ __forceinline__ void skinny_strip(const uint16_t* __restrict__ x, int64_t xs,
                                             const uint16_t* __restrict__ w, uint16_t* __restrict__ out,
                                             int M, int N, int K, int act, int strip,
                                             SkinnyRed<MF, GU, WV>& sums) {
    constexpr int RT = GU ? 2 : 1;
    auto& red = sums.at;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int r = lane & 15, q = lane >> 4;
    const int n0 = strip * 16;
    const int st = K / 32;
    const int k0 = wid * st / WV, kn = (wid + 1) * st / WV - k0;     // the wave's steps

    const uint16_t* wp[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        const int row = min(n0 + r, N - 1) + (t ? N : 0);
        wp[t] = w + (size_t)row * K + (size_t)k0 * 32 + q * 8;
    }
    const uint16_t* xp[MF];
#pragma unroll
    for (int f = 0; f < MF; ++f)
        xp[f] = x + (size_t)min(f * 16 + r, M - 1) * xs + (size_t)k0 * 32 + q * 8;

    sk_f4 acc[RT][MF];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int f = 0; f < MF; ++f) acc[t][f] = sk_f4{0.0f, 0.0f, 0.0f, 0.0f};
    sk_u4 wb[D][RT], xb[D][MF];
    auto load = [&](int p, int k) {
#pragma unroll
        for (int t = 0; t < RT; ++t) wb[p][t] = *reinterpret_cast<const sk_u4*>(wp[t] + (size_t)k * 32);
#pragma unroll
        for (int f = 0; f < MF; ++f) xb[p][f] = *reinterpret_cast<const sk_u4*>(xp[f] + (size_t)k * 32);
    };
    auto mul = [&](int p) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int f = 0; f < MF; ++f)
                acc[t][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(sk_b8, wb[p][t]), __builtin_bit_cast(sk_b8, xb[p][f]), acc[t][f], 0, 0, 0);
    };
    // rounds of D steps, the next round's loads issued as registers come free; the
    // last round is apart so that every wait counts exactly
    const int rounds = kn / D;
    if (rounds > 0) {
#pragma unroll
        for (int p = 0; p < D; ++p) load(p, p);
        for (int i = 1; i < rounds; ++i) {
#pragma unroll
            for (int p = 0; p < D; ++p) {
                mul(p);
                load(p, i * D + p);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int p = 0; p < D; ++p) mul(p);
    }
    for (int k = rounds * D; k < kn; ++k) {
        load(0, k);
        mul(0);
    }

    // lane: activation row r of a fragment, weight rows q * 4 .. + 3
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int f = 0; f < MF; ++f)
            *reinterpret_cast<sk_f4*>(&red[wid][t][f][r][q * 4]) = acc[t][f];
    __syncthreads();
    for (int i = tid; i < MF * 256; i += WV * 64) {
        const int c = i & 15, m = (i >> 4) & 15, f = i >> 8;
        const int row = f * 16 + m, n = n0 + c;
        if (row >= M || n >= N) continue;
        float a = 0.0f, b = 0.0f;
#pragma unroll
        for (int v = 0; v < WV; ++v) {
            a += red[v][0][f][m][c];
            if (GU) b += red[v][RT - 1][f][m][c];
        }
        out[(size_t)row * N + n] = f32_to_bf16(GU ? sk_gate(a, act) * b : a);
    }
}
