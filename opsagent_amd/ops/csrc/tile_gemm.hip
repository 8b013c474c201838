// Products of more than 128 rows: C[M, N] = x[M, K] W[N, K]^T in bf16, plain, gate-up with its
// activation, or as float32 column parts, and in e4m3 with a scale a row of both.
//
// Three things bound them, measured apart on 2048 x 8192 x 4096 in tiles of 256 x 256. The matrix
// cores take 1.05 us a step of 64 columns on random operands that LDS feeds (1.75 PFLOP/s; 2.4 on
// zeros: power, not issue). The LDS reads of a step take 0.64 us. And the transfers into LDS stop at
// 64 KB under way a CU, whatever the depth of the ring: 150 GB/s a CU from the L2, 110 where x and
// W lie in the cache before memory, 65 where W comes from memory, which is 1 us a step. So small
// tiles are bound by transfers (128 x 128 runs at 1.3 PFLOP/s without them, at 0.9 with) and large
// ones by power, and what is won lies in tiles that fill the CUs. Two groups of four waves, a wave of
// each on every SIMD, therefore take turns: while one reads its fragments from LDS and sends for a
// later step, the other multiplies; a barrier ends each phase. Us, the library (gate-up: and the
// activation kernel) / here (splits: and the sum): 4096 x 14336, M = 130 55 / 36, 512 91 / 67, 800
// 124 / 94, 2048 206 / 183; 4096 x 4096, 800 39 / 34, 2048 59 / 56; 6144 x 4096, 130 40 / 24, 700 49 /
// 41, 2048 82 / 84; 2048 x 8192, 256 28 / 24, 1024 50 / 48, 2048 72 / 68; gate-up 2 x 14336 x 4096, 130
// 63 / 58, 800 189 / 167, 2048 391 / 366; 2 x 2816 x 2048, 512 29 / 22, 1434 52 / 35.
// Slower: transfers in turn with the LDS reads or between the products; four waves of 128 x 128 (the
// compiler copies sums between register files); v_mfma_f32_32x32x16_bf16 (1.6 PFLOP/s from LDS);
// touching the lines of later steps (results come in order: it waits behind them).
#include <algorithm>
#include <type_traits>

#include "common.h"

typedef __attribute__((ext_vector_type(4))) float tgf4;
typedef __attribute__((ext_vector_type(8))) short tgs8;
typedef __attribute__((ext_vector_type(8))) int tgi8;
typedef __attribute__((ext_vector_type(16))) float tgf16;

// A fragment's 16 rows of a step: 128 bytes of each, 32 a lane. Lane group c has chunks c and c + 4, the
// columns of the two products that they stand for.
struct TgFrag {
    tgs8 b[2];
};
struct TgAt {
    int a, b;
    __device__ __forceinline__ TgAt(int lane) {
        const int r = lane & 15, c = lane >> 4;
        a = r * 128 + ((c ^ (r >> 1)) << 4);
        b = r * 128 + (((c + 4) ^ (r >> 1)) << 4);
    }
};

// the fragments of FI x FJ over a step
template <int FI, int FJ>
__device__ __forceinline__ void tg_multiply(tgf4 (&acc)[FI][FJ], const TgFrag (&wf)[FJ], const TgFrag (&xf)[FI]) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int i = 0; i < FI; ++i)
#pragma unroll
            for (int j = 0; j < FJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j].b[k], xf[i].b[k], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
}
template <int FI, int FJ>
__device__ __forceinline__ void tg_read(TgFrag (&wf)[FJ], TgFrag (&xf)[FI], const char* wr, const char* xr, const TgAt& at) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
        for (int j = 0; j < FJ; ++j) wf[j].b[k] = *reinterpret_cast<const tgs8*>(wr + j * 2048 + (k ? at.b : at.a));
#pragma unroll
        for (int i = 0; i < FI; ++i) xf[i].b[k] = *reinterpret_cast<const tgs8*>(xr + i * 2048 + (k ? at.b : at.a));
    }
    __builtin_amdgcn_sched_barrier(0);
}

// e4m3: fragments of 32 rows, two products of 64 columns a step with unit block scales (the only fp8
// products past the bf16 rate). Lane half h has bytes 64 k + 32 h and up of its row: products, order
// and rounding of the one-barrier tiles (fp8_moe.hip), since an 8-bit model turns another order of the
// sums into 0.01 to 0.03 of its activations. v_mfma_scale_f32_16x16x128 gains 2% more (28672 x 4096,
// M = 700 93.4 us, here 94).
struct TgFrag8 {
    tgi8 k[2];
};
struct TgAt8 {
    int at[2][2];
    __device__ __forceinline__ TgAt8(int lane) {
        const int r = lane & 31, h = lane >> 5;
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int c = 0; c < 2; ++c) at[k][c] = r * 128 + (((k * 4 + h * 2 + c) ^ (r >> 1 & 7)) << 4);
    }
};
template <int FI, int FJ>
__device__ __forceinline__ void tg_read(TgFrag8 (&wf)[FJ], TgFrag8 (&xf)[FI], const char* wr, const char* xr, const TgAt8& at) {
    auto one = [&](const char* rows, int k) {
        union {
            uint4 c[2];
            tgi8 v;
        } f;
        f.c[0] = *reinterpret_cast<const uint4*>(rows + at.at[k][0]);
        f.c[1] = *reinterpret_cast<const uint4*>(rows + at.at[k][1]);
        return f.v;
    };
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
        for (int j = 0; j < FJ; ++j) wf[j].k[k] = one(wr + j * 4096, k);
#pragma unroll
        for (int i = 0; i < FI; ++i) xf[i].k[k] = one(xr + i * 4096, k);
    }
    __builtin_amdgcn_sched_barrier(0);
}
template <int FI, int FJ>
__device__ __forceinline__ void tg_multiply(tgf16 (&acc)[FI][FJ], const TgFrag8 (&wf)[FJ], const TgFrag8 (&xf)[FI]) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int i = 0; i < FI; ++i)
#pragma unroll
            for (int j = 0; j < FJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wf[j].k[k], xf[i].k[k], acc[i][j], 0, 0, 0, 0x7f, 0, 0x7f);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
}

// The step of its columns that a strip of weight rows starts at, to go round them: rows a few KiB apart
// lie on the same memory channels, and blocks that read the same columns share those. Few rows of x
// wait for it, us together / apart: gate-up 2 x 14336 x 4096, M = 130 61 / 57, 200 69 / 65, 333 81 / 78;
// 32000 x 4096, 130 63 / 52, 200 68 / 61; 4096 x 4096, 130 19.8 / 17.2. More tiles of rows are bound by other
// things, and what they share of x is read again by strips apart (2048 x 8192, 2000 69 / 74).
__device__ __forceinline__ int tg_turned(int strip, int steps, int mtiles) {
    return mtiles > 2 ? 0 : (strip >> 1) * 3 % steps;
}

template <int V>
__device__ __forceinline__ void tg_wait() {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(V) : "memory");
}

__device__ __forceinline__ void tg_read_done() {
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
}

__device__ __forceinline__ void tg_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" : : : "memory");
    __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ float tg_gate(float g, float u, int act) {
    if (act == 2) {
        const float t = 0.7978845608028654f * fmaf(0.044715f * g * g, g, g);
        return 0.5f * g * (1.0f + tanhf(t)) * u;
    }
    return g / (1.0f + __expf(-g)) * u;
}

// the weight row (from the strip's first on) that LDS row b of the strip holds: a wave's fragments in
// pairs whose lanes hold eight neighbouring outputs together, gate rows beside their up rows
template <int FJ, bool GU, bool F8 = false>
__device__ __forceinline__ int tg_wrow(int b) {
    static_assert(FJ % 2 == 0, "pairs");
    // a lane's eights together; gate-up: a wave's two fragments are 32 gate rows and their up rows
    if (F8) return (GU ? (b >> 6) * 32 + (b & 16) : b & ~15) + (b >> 2 & 1) * 8 + (b >> 3 & 1) * 4 + (b & 3);
    const int wv = b / (16 * FJ), j = b / 16 % FJ, r = b & 15;
    if (GU) {
        if (FJ % 4 == 0) return wv * FJ * 8 + (j >> 2) * 32 + (r >> 2) * 8 + (j & 1) * 4 + (r & 3);
        return wv * FJ * 8 + (j >> 1) * 16 + r;
    }
    return wv * FJ * 16 + (j >> 1) * 32 + (r >> 2) * 8 + (j & 1) * 4 + (r & 3);
}
template <int FJ, bool GU, bool F8 = false>
__device__ __forceinline__ bool tg_isup(int b) {
    if (F8) return GU && (b & 32);
    const int j = b / 16 % FJ;
    return GU && (FJ % 4 == 0 ? (j >> 1 & 1) : (j & 1));
}

// fragments I0 .. I1 of a wave whose first row is row0
template <int FI, int FJ, bool GU, int I0, int I1>
__device__ __forceinline__ void tg_store(tgf4 (&acc)[FI][FJ], uint16_t* out, float* part, int row0, int n0, int wc, int M, int N, int sp, int act) {
    const int fr = threadIdx.x & 15, fc = threadIdx.x >> 4 & 3;
    // D: column (row of x) lane & 15, rows (weight rows) (lane >> 4) * 4 and up
#pragma unroll
    for (int i = I0; i < I1; ++i) {
        const int row = row0 + i * 16 + fr;
        if (row >= M) continue;
        if (GU) {
#pragma unroll
            for (int j = 0; j < FJ; j += (FJ % 4 == 0 ? 4 : 2)) {
                constexpr int V = FJ % 4 == 0 ? 2 : 1;
                const int col = n0 + wc * FJ * 8 + (V == 2 ? (j >> 2) * 32 + fc * 8 : (j >> 1) * 16 + fc * 4);
                if (col >= N) continue;
                uint32_t o[2 * V];
#pragma unroll
                for (int v = 0; v < V; ++v)
#pragma unroll
                    for (int e = 0; e < 2; ++e)
                        o[v * 2 + e] = pack_bf16x2(tg_gate(acc[i][j + v][2 * e], acc[i][j + V + v][2 * e], act),
                                                   tg_gate(acc[i][j + v][2 * e + 1], acc[i][j + V + v][2 * e + 1], act));
                if constexpr (V == 2)
                    *reinterpret_cast<uint4*>(out + (size_t)row * N + col) = make_uint4(o[0], o[1], o[2], o[3]);
                else
                    *reinterpret_cast<uint2*>(out + (size_t)row * N + col) = make_uint2(o[0], o[1]);
            }
            continue;
        }
#pragma unroll
        for (int j = 0; j < FJ; ++j) {
            const int col = n0 + tg_wrow<FJ, false>((wc * FJ + j) * 16 + fc * 4);
            if (col >= N) continue;
            if (part) {
                *reinterpret_cast<tgf4*>(part + ((int64_t)sp * M + row) * N + col) = acc[i][j];
                continue;
            }
            if (j % 2) continue;
            *reinterpret_cast<uint4*>(out + (size_t)row * N + col) =
                make_uint4(pack_bf16x2(acc[i][j][0], acc[i][j][1]), pack_bf16x2(acc[i][j][2], acc[i][j][3]),
                           pack_bf16x2(acc[i][j + 1][0], acc[i][j + 1][1]),
                           pack_bf16x2(acc[i][j + 1][2], acc[i][j + 1][3]));
        }
    }
}

// 32 x 32 fragments: column (row of x) lane & 31, a lane half twice eight weight rows beside the other's
template <int FI, int FJ>
__device__ __forceinline__ void tg_store8(const tgf16 (&acc)[FI][FJ], const float* xscale, const float* wscale,
                                          uint16_t* out, int row0, int n0, int wc, int M, int N) {
    const int fr = threadIdx.x & 31, half = threadIdx.x >> 5 & 1;
#pragma unroll
    for (int i = 0; i < FI; ++i) {
        const int row = row0 + i * 32 + fr;
        if (row >= M) continue;
        const float sx = xscale[row];
#pragma unroll
        for (int j = 0; j < FJ; ++j)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int col = n0 + (wc * FJ + j) * 32 + c * 16 + half * 8;
                if (col >= N) continue;                       // N % 8 == 0
                uint32_t o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int k = c * 8 + 2 * e;
                    o[e] = pack_bf16x2(acc[i][j][k] * sx * wscale[col + 2 * e], acc[i][j][k + 1] * sx * wscale[col + 2 * e + 1]);
                }
                *reinterpret_cast<uint4*>(out + (size_t)row * N + col) = make_uint4(o[0], o[1], o[2], o[3]);
            }
    }
}

// gate-up: the rows of silu(gate) * up that the quantizer of two bf16 halves would make of the plain product,
// bit for bit, at half of its bytes. Us for 700 rows of 2 x 14336 x 4096, product and quantizer: 98 + 14 / 98 + 7;
// a prompt of four layers 1069 -> 1043.
template <int FI>
__device__ __forceinline__ void tg_store8_gate(const tgf16 (&acc)[FI][2], const float* xscale, const float* wscale,
                                               uint16_t* out, int row0, int n0, int wc, int M, int N) {
    const int fr = threadIdx.x & 31, half = threadIdx.x >> 5 & 1;
#pragma unroll
    for (int i = 0; i < FI; ++i) {
        const int row = row0 + i * 32 + fr;
        if (row >= M) continue;
        const float sx = xscale[row];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int col = n0 + wc * 32 + c * 16 + half * 8;
            if (col >= N) continue;                           // N % 8 == 0
            uint32_t o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int k = c * 8 + 2 * e;
                const float* sg = wscale + col + 2 * e;
                const float* su = sg + N;
                o[e] = silu_mul_bf16x2(pack_bf16x2(acc[i][0][k] * sx * sg[0], acc[i][0][k + 1] * sx * sg[1]),
                                       pack_bf16x2(acc[i][1][k] * sx * su[0], acc[i][1][k + 1] * sx * su[1]));
            }
            *reinterpret_cast<uint4*>(out + (size_t)row * N + col) = make_uint4(o[0], o[1], o[2], o[3]);
        }
    }
}

// Tiles of 32 FI x 64 FJ: group 0 takes the upper half of the rows, group 1 the lower, a wave a quarter of
// the columns. Phase 2 t: group 0 reads step t and group 1 multiplies step t - 1; phase 2 t + 1: group
// 1 reads step t. Group 0 sends for x, XS steps deep, group 1 for W, WS deep: W comes from further away.
// What phase 2 t sends for takes the place of step t - 1, which both have read. A wave waits for its own
// transfers before the barrier that lets step t + 1 be read.
//
// Both operands come by 16-byte global_load_lds, inline asm: hipcc's own waits drain builtin transfers
// before the first LDS read. 16-byte chunk c of row r lies at c ^ (r >> 1 & 7): the 16 rows of a fragment
// read touch every bank once. Rows past M and weight rows past N repeat the last one. Work items go to the
// dies in runs, the row tiles of a strip of weight rows next to each other.
template <int FI, int FJ, int XS, int WS, bool GU, bool F8>
__global__ __launch_bounds__(512, 2) void tile_gemm_kernel(
    const char* __restrict__ x, int64_t xs, const char* __restrict__ w,
    const float* __restrict__ xscale, const float* __restrict__ wscale, uint16_t* __restrict__ out, float* __restrict__ part, int M, int N, int64_t kb, int mtiles,
    int splits, int items, int act) {
    constexpr int BM = 32 * FI, BN = 64 * FJ;
    constexpr int XB = BM * 128, WB = BN * 128;      // bytes of a step
    constexpr int LP = FI > 2 * FJ ? FI : 2 * FJ;    // transfers of a wave and step, at most
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int per = gridDim.x >> 3;
    const int item = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (item >= items) return;
    const int strip = item / (splits * mtiles), rest = item - strip * splits * mtiles;
    const int sp = rest / mtiles, m0 = (rest - sp * mtiles) * BM;
    const int n0 = strip * (GU ? BN / 2 : BN);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = wave >> 2, wc = wave & 3;
    const int steps = (int)(kb / 128);                // kb: bytes of a weight row, xs: of a row of x
    const int s0 = (int)((int64_t)steps * sp / splits), s1 = (int)((int64_t)steps * (sp + 1) / splits);
    const int n = s1 - s0;

    const int turned = F8 ? 0 : tg_turned(strip, n, mtiles);
    int ahead = n - turned;                          // steps to the last column
    // transfers of eight rows: group 0 those of x, group 1 those of w
    const char* base = grp ? w + (int64_t)n0 * kb + (int64_t)(s0 + turned) * 128
                           : x + (int64_t)m0 * xs + (int64_t)(s0 + turned) * 128;
    uint32_t off[LP];
#pragma unroll
    for (int p = 0; p < LP; ++p) {
        const int r = (p * 4 + wc) * 8 + (lane >> 3);
        const int chunk = ((lane & 7) ^ (r >> 1 & 7)) * 16;
        if (!grp) off[p] = (uint32_t)min(r, M - 1 - m0) * (uint32_t)xs + chunk;
        else off[p] = (uint32_t)(min(tg_wrow<FJ, GU, F8>(r), N - 1 - n0) + (tg_isup<FJ, GU, F8>(r) ? N : 0)) * (uint32_t)kb + chunk;
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem + (grp ? XS * XB : 0) + wc * 1024);
    auto stage_x = [&](int buf) {
#pragma unroll
        for (int p = 0; p < FI; ++p) lds_transfer16(lds0 + buf * XB + p * 4096, off[p], base);
        base += 128;
        if (!F8 && --ahead == 0) base -= (int64_t)n * 128;
    };
    auto stage_w = [&](int buf) {
#pragma unroll
        for (int p = 0; p < 2 * FJ; ++p) lds_transfer16(lds0 + buf * WB + p * 4096, off[p], base);
        base += 128;
        if (!F8 && --ahead == 0) base -= (int64_t)n * 128;
    };
    // this wave's transfers of the step that `behind` younger ones follow
    auto landed_x = [&](int behind) {
        if (XS > 3 && behind >= 2) tg_wait<2 * FI>();
        else if (XS > 2 && behind >= 1) tg_wait<FI>();
        else tg_wait<0>();
    };
    auto landed_w = [&](int behind) {
        if (WS > 3 && behind >= 2) tg_wait<4 * FJ>();
        else if (WS > 2 && behind >= 1) tg_wait<2 * FJ>();
        else tg_wait<0>();
    };

    constexpr int AI = F8 ? FI / 2 : FI, AJ = F8 ? FJ / 2 : FJ;
    static_assert(!F8 || (FI % 2 == 0 && (!GU || FJ == 4)), "fragments of 32 rows, gate-up in pairs");
    std::conditional_t<F8, tgf16, tgf4> acc[AI][AJ] = {};
    if (!grp) {
#pragma unroll
        for (int t = 0; t < XS - 1; ++t)
            if (t < n) stage_x(t);
        landed_x(min(XS - 2, n - 1));
        tg_barrier();
    } else {
#pragma unroll
        for (int t = 0; t < WS - 1; ++t)
            if (t < n) stage_w(t);
        landed_w(min(WS - 2, n - 1));
        tg_barrier();
        tg_barrier();
    }
    const std::conditional_t<F8, TgAt8, TgAt> at(lane);
    int xbuf = 0, wbuf = 0;
    for (int t = 0; t < n; ++t) {
        const char* xr = smem + xbuf * XB + grp * FI * 16 * 128;
        const char* wr = smem + XS * XB + wbuf * WB + wc * FJ * 16 * 128;
        std::conditional_t<F8, TgFrag8, TgFrag> xf[AI], wf[AJ];
        tg_read<AI, AJ>(wf, xf, wr, xr, at);
        if (!grp) {
            if (t + XS - 1 < n) stage_x(xbuf == 0 ? XS - 1 : xbuf - 1);
        } else {
            if (t + WS - 1 < n) stage_w(wbuf == 0 ? WS - 1 : wbuf - 1);
            landed_w(min(WS - 2, n - 2 - t));
        }
        tg_read_done();
        tg_barrier();
        tg_multiply<AI, AJ>(acc, wf, xf);
        if (!grp) landed_x(min(XS - 2, n - 2 - t));
        tg_barrier();
        xbuf = xbuf + 1 == XS ? 0 : xbuf + 1;
        wbuf = wbuf + 1 == WS ? 0 : wbuf + 1;
    }
    if (!grp) tg_barrier();

    const int row0 = m0 + grp * FI * 16;
    if constexpr (F8 && GU) tg_store8_gate<AI>(acc, xscale, wscale, out, row0, n0, wc, M, N);
    else if constexpr (F8) tg_store8<AI, AJ>(acc, xscale, wscale, out, row0, n0, wc, M, N);
    else tg_store<FI, FJ, GU, 0, FI>(acc, out, part, row0, n0, wc, M, N, sp, act);
}

// Tiles of 32 FI x 32 FJ: a wave of 2 x 2 takes a quarter of the tile and the groups take the steps in
// turn, each into sums of its own, which are added up at the end. A quarter a wave reads less LDS than
// an eighth (128 x 128: 64 KB a step and not 98), and a phase is a whole step for both (800 x 4096 x 4096
// 40 us with eighths, 34 here; 800 x 4096 x 14336 126, 103).
template <int FI, int FJ, int ST, bool GU>
__global__ __launch_bounds__(512, 2) void tile_gemm_turns_kernel(
    const char* __restrict__ x, int64_t xs, const char* __restrict__ w,
    const float* __restrict__ xscale, const float* __restrict__ wscale, uint16_t* __restrict__ out, float* __restrict__ part, int M, int N, int64_t kb, int mtiles,
    int splits, int items, int act) {
    constexpr int BM = 32 * FI, BN = 32 * FJ;
    constexpr int STEP = (BM + BN) * 128, LP = FI + FJ;      // transfers of a wave: FI of x, FJ of w
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int per = gridDim.x >> 3;
    const int item = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (item >= items) return;
    const int strip = item / (splits * mtiles), rest = item - strip * splits * mtiles;
    const int sp = rest / mtiles, m0 = (rest - sp * mtiles) * BM;
    const int n0 = strip * (GU ? BN / 2 : BN);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = wave >> 2, wid = wave & 3, wm = wid >> 1, wc = wid & 1;
    const int steps = (int)(kb / 128);                // kb: bytes of a weight row, xs: of a row of x
    const int s0 = (int)((int64_t)steps * sp / splits), s1 = (int)((int64_t)steps * (sp + 1) / splits);
    const int n = s1 - s0;

    const char* xb = x + (int64_t)m0 * xs + (int64_t)s0 * 128;
    const char* wb = w + (int64_t)n0 * kb + (int64_t)s0 * 128;
    uint32_t off[LP];
#pragma unroll
    for (int p = 0; p < LP; ++p) {
        const int r = ((p < FI ? p : p - FI) * 4 + wid) * 8 + (lane >> 3);
        const int chunk = ((lane & 7) ^ (r >> 1 & 7)) * 16;
        if (p < FI) off[p] = (uint32_t)min(r, M - 1 - m0) * (uint32_t)xs + chunk;
        else off[p] = (uint32_t)(min(tg_wrow<FJ, GU>(r), N - 1 - n0) + (tg_isup<FJ, GU>(r) ? N : 0)) * (uint32_t)kb + chunk;
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem + wid * 1024);
    const int turned = tg_turned(strip, n, mtiles);
    auto stage = [&](int step, int buf) {
        const int at = step + turned < n ? step + turned : step + turned - n;
        const char* xt = xb + (int64_t)at * 128;
        const char* wt = wb + (int64_t)at * 128;
#pragma unroll
        for (int p = 0; p < LP; ++p) lds_transfer16(lds0 + buf * STEP + p * 4096, off[p], p < FI ? xt : wt);
    };
    // Phase p: group p & 1 reads step p and sends for step p + ST - 1, into the place of step p - 1,
    // while the other multiplies step p - 1. Step s is sent for by group (s + ST - 1) & 1, which
    // waits for it at the end of phase s - 1: after reading (ST even) or after multiplying.
    constexpr int OWN = (ST - 1) & 1;
    auto landed = [&](int s) {
        const int young = (min(s + ST - 2, n - 1) - s) / 2;     // younger steps of this group under way
        if (ST > 5 && young >= 2) tg_wait<2 * LP>();
        else if (ST > 3 && young >= 1) tg_wait<LP>();
        else tg_wait<0>();
    };
#pragma unroll
    for (int t = 0; t < ST - 1; ++t)
        if (((t + OWN) & 1) == grp && t < n) stage(t, t);
    if (grp == OWN) landed(0);
    tg_barrier();
    if (grp) {
        if (ST % 2 && n > 1) landed(1);
        tg_barrier();
    }
    tgf4 acc[FI][FJ] = {};
    const TgAt at(lane);
    int buf = grp;
    for (int s = grp; s < n; s += 2) {
        const char* xr = smem + buf * STEP + wm * FI * 2048;
        const char* wr = smem + buf * STEP + BM * 128 + wc * FJ * 2048;
        TgFrag xf[FI], wf[FJ];
        tg_read<FI, FJ>(wf, xf, wr, xr, at);
        if (s + ST - 1 < n) stage(s + ST - 1, buf == 0 ? ST - 1 : buf - 1);
        if (ST % 2 == 0 && s + 1 < n) landed(s + 1);
        tg_read_done();
        tg_barrier();                                        // the end of phase s
        tg_multiply<FI, FJ>(acc, wf, xf);
        if (s + 1 < n) {
            if (ST % 2 && s + 2 < n) landed(s + 2);
            tg_barrier();                                    // the end of phase s + 1
        }
        buf = buf + 2 >= ST ? buf + 2 - ST : buf + 2;
    }
    // each group takes the other's sums of half of its fragments
    constexpr int FH = (FI + 1) / 2;
    tgf4* ex = reinterpret_cast<tgf4*>(smem);
    if (grp) {
#pragma unroll
        for (int i = 0; i < FH; ++i)
#pragma unroll
            for (int j = 0; j < FJ; ++j) ex[((i * FJ + j) * 4 + wid) * 64 + lane] = acc[i][j];
    } else {
#pragma unroll
        for (int i = FH; i < FI; ++i)
#pragma unroll
            for (int j = 0; j < FJ; ++j) ex[((i * FJ + j) * 4 + wid) * 64 + lane] = acc[i][j];
    }
    __syncthreads();
    if (grp) {
#pragma unroll
        for (int i = FH; i < FI; ++i)
#pragma unroll
            for (int j = 0; j < FJ; ++j) acc[i][j] += ex[((i * FJ + j) * 4 + wid) * 64 + lane];
        tg_store<FI, FJ, GU, FH, FI>(acc, out, part, m0 + wm * FI * 16, n0, wc, M, N, sp, act);
    } else {
#pragma unroll
        for (int i = 0; i < FH; ++i)
#pragma unroll
            for (int j = 0; j < FJ; ++j) acc[i][j] += ex[((i * FJ + j) * 4 + wid) * 64 + lane];
        tg_store<FI, FJ, GU, 0, FH>(acc, out, part, m0 + wm * FI * 16, n0, wc, M, N, sp, act);
    }
}

// Forms, and what they take in us: a step (64 columns, e4m3 128), more of it when all CUs work (power, and
// x from beside the chip), starting and ending a tile; least squares over 2700 times of 110 products
// (e4m3: 460 of 104), to 6 to 11% (6%). The choice by them takes 1.01 of the time of the best form (1.13 at
// most). e4m3 has forms of the first kernel only: the turns of the second and column splits add up in
// another order, and an 8-bit model turns that into 0.01 to 0.03 of its activations.
struct TgForm {
    int id, bm, bn;
    float step, more, tile;
};
static const TgForm tg_forms[] = {
    {0, 256, 256, 0.872f, 0.498f, 9.2f}, {1, 224, 256, 0.796f, 0.425f, 8.3f}, {2, 192, 256, 0.734f, 0.381f, 7.6f},
    {3, 160, 256, 0.673f, 0.295f, 7.2f}, {4, 256, 128, 0.531f, 0.295f, 6.7f}, {5, 224, 128, 0.471f, 0.264f, 6.1f},
    {6, 160, 128, 0.393f, 0.201f, 5.3f}, {7, 128, 128, 0.352f, 0.195f, 4.1f}, {8, 96, 128, 0.292f, 0.170f, 2.8f},
    {9, 128, 64, 0.259f, 0.116f, 2.5f},
};
static const TgForm tg_forms8[] = {
    {0, 256, 256, 1.063f, 0.734f, 6.6f}, {1, 192, 256, 0.887f, 0.539f, 5.3f}, {2, 128, 256, 0.583f, 0.349f, 5.6f},
    {3, 192, 128, 0.525f, 0.227f, 5.3f}, {4, 64, 128, 0.396f, 0.066f, 3.5f},
};

// The fastest of the forms and column splits as form * 256 + splits, and its time in *us. A split has eight steps.
template <int FORMS>
static int tg_choose(const TgForm (&forms)[FORMS], int M, int rows, int steps, bool split, bool summed, float* us_best) {
    const float mn = (float)M * rows;
    float best = 1e30f;
    int plan = -1;
    for (const TgForm& t : forms) {
        const int64_t tiles = (int64_t)CEIL_DIV(M, t.bm) * CEIL_DIV(rows, t.bn);
        const int most = split && tiles < 256 ? (int)std::min<int64_t>(8, 256 / tiles) : 1;
        for (int sp = 1; sp <= most && (sp == 1 || steps / sp >= 8); ++sp) {
            const int64_t blocks = tiles * sp, full = blocks / 256, rest = blocks % 256;
            const float n = (float)steps / sp;
            float us = full * (n * (t.step + t.more) + 0.6f * t.tile) + 0.4f * t.tile + 2;
            if (rest) us += n * (t.step + t.more * rest / 256) + 0.6f * t.tile;
            if (sp > 1) us += sp * mn * 0.36e-6f + (summed ? (sp * 4 - 2) * mn / 4.5e6f : 2.5f + sp * mn * 4 / 4.5e6f);
            if (us < best) best = us, plan = t.id * 256 + sp;
        }
    }
    *us_best = best;
    return plan;
}

// A lane's place in a tile is 32 bits wide: rows of x less than 8 MB apart, and the weight rows of a strip
// (gate-up: and their up rows, N further on) within 4 GB
static bool tg_within(int64_t xs, int64_t N, int64_t K, bool gateup) {
    return xs < (1 << 22) && ((gateup ? N : 0) + 256) * K * 2 < ((int64_t)1 << 32);
}

// The plan of M rows, N (gate-up: 2 N) weight rows and K columns; -1 for sizes that the product does not
// take, and for gate-up products that other forms take sooner. Splits fill the CUs where the tiles leave
// some idle, at most one block a CU; their parts are written, and read again by a kernel of their own (4.5
// TB/s, 2.5 us) or, summed, by a norm that would have read the product. Gate-up does not split: where
// splits and an activation kernel would be the faster way (2 x 2048 x 8192, M = 246 50.9 us in one, 38.4
// the library and the kernel) it is left to them.
extern "C" int oa_tile_gemm_plan(int M, int N, int K, int gateup, int summed) {
    if (M < 1 || N < 8 || N % 8 != 0 || N > (1 << 29) || K < 512 || K % 64 != 0) return -1;
    if (!tg_within(K, N, K, gateup)) return -1;
    float one, two;
    if (!gateup) return tg_choose(tg_forms, M, N, K / 64, true, summed, &one);
    const int plan = tg_choose(tg_forms, M, 2 * N, K / 64, false, false, &one);
    tg_choose(tg_forms, M, 2 * N, K / 64, true, false, &two);
    return one > two + 3 + (float)M * N * 6 / 4.5e6f ? -1 : plan;
}

extern "C" double oa_gemm_fp8_us(int M, int N, int K);

// The form of an e4m3 product, -1 for sizes that it does not take and where the one-barrier tiles
// (fp8_moe.hip), which answer the same bit for bit, are the faster ones by both models (they are late by 6%
// here): at 84 sizes of 130 to 2048 rows this takes 0.929 of the time of those, 0.926 would be the best. Us,
// those / here: 28672 x 4096, M = 130 41.6 / 36.6, 700 109.6 / 94.7, 1700 228 / 193, 2048 259 / 236; 6144 x
// 4096, 700 33.6 / 28.2, 1400 56.3 / 44.4; 4096 x 14336, 1400 110 / 88; 2048 x 2048, 450 13.2 / 12.1; 16384
// x 2048, 450 25.7 / 23.4; but 6144 x 4096, 450 21.5 / 26.9 and 2048 x 8192, 1400 34.8 / 45.6.
extern "C" int oa_tile_gemm_fp8_form(int M, int N, int K) {
    if (M < 1 || N < 8 || N % 8 != 0 || N > (1 << 29) || K < 512 || K % 128 != 0 || K >= (1 << 23)) return -1;
    float us;
    const int plan = tg_choose(tg_forms8, M, N, K / 128, false, false, &us);
    return us < 1.06 * oa_gemm_fp8_us(M, N, K) ? plan >> 8 : -1;
}

extern "C" int oa_ring_sum(void* stream, const void* part, void* out, int M, int N, int splits);

// xs, kb: bytes of a row of x and of a weight row
static int tg_run(hipStream_t s, const void* x, int64_t xs, const void* w, const void* xscale, const void* wscale,
                  void* out, void* part, int M, int N, int64_t kb, int form, int splits, int act, bool f8) {
#define TG_LAUNCH(kernel, BM, BN, lds)                                                             \
    do {                                                                                           \
        const int mt = CEIL_DIV(M, BM);                                                            \
        const int64_t items = (int64_t)CEIL_DIV(N, (BN) / (act ? 2 : 1)) * mt * splits;            \
        if (items > (1 << 28)) return -103;                                                        \
        hipLaunchKernelGGL(kernel, dim3((unsigned)(CEIL_DIV(items, 8) * 8)), dim3(512), lds, s,    \
                           (const char*)x, xs, (const char*)w, (const float*)xscale,               \
                           (const float*)wscale, (uint16_t*)out, (float*)part, M, N, kb, mt,       \
                           splits, (int)items, act);                                               \
    } while (0)
#define TG_HALVES(FI, FJ, XS, WS, GU, F8)                                                        \
    TG_LAUNCH((tile_gemm_kernel<FI, FJ, XS, WS, GU, F8>), 32 * (FI), 64 * (FJ), ((XS) * 32 * (FI) + (WS) * 64 * (FJ)) * 128)
#define TG_WIDE(FI, XS)                                  \
    do {                                                 \
        if (act) TG_HALVES(FI, 4, XS, 3, true, false);   \
        else TG_HALVES(FI, 4, XS, 3, false, false);      \
    } while (0)
#define TG_TURNS(FI, FJ, ST)                                                                             \
    do {                                                                                                 \
        constexpr int lds = (ST) * 32 * ((FI) + (FJ)) * 128;                                             \
        if (act) TG_LAUNCH((tile_gemm_turns_kernel<FI, FJ, ST, true>), 32 * (FI), 32 * (FJ), lds);       \
        else TG_LAUNCH((tile_gemm_turns_kernel<FI, FJ, ST, false>), 32 * (FI), 32 * (FJ), lds);          \
    } while (0)
    if (f8 && act) {
        switch (form) {
            case 0: TG_HALVES(8, 4, 2, 3, true, true); break;
            case 1: TG_HALVES(6, 4, 2, 3, true, true); break;
            case 2: TG_HALVES(4, 4, 3, 3, true, true); break;
            default: return -105;
        }
        HIP_CHECK_LAUNCH();
        return 0;
    }
    if (f8) {
        switch (form) {
            case 0: TG_HALVES(8, 4, 2, 3, false, true); break;
            case 1: TG_HALVES(6, 4, 2, 3, false, true); break;
            case 2: TG_HALVES(4, 4, 3, 3, false, true); break;
            case 3: TG_HALVES(6, 2, 3, 4, false, true); break;
            case 4: TG_HALVES(2, 2, 4, 4, false, true); break;
            default: return -105;
        }
        HIP_CHECK_LAUNCH();
        return 0;
    }
    switch (form) {
        case 0: TG_WIDE(8, 2); break;
        case 1: TG_WIDE(7, 2); break;
        case 2: TG_WIDE(6, 2); break;
        case 3: TG_WIDE(5, 3); break;
        case 4: TG_TURNS(8, 4, 3); break;
        case 5: TG_TURNS(7, 4, 3); break;
        case 6: TG_TURNS(5, 4, 4); break;
        case 7: TG_TURNS(4, 4, 4); break;
        case 8: TG_TURNS(3, 4, 5); break;
        case 9: TG_TURNS(4, 2, 6); break;
        default: return -105;
    }
#undef TG_TURNS
#undef TG_WIDE
#undef TG_HALVES
#undef TG_LAUNCH
    HIP_CHECK_LAUNCH();
    return 0;
}

// out [M, N] = x [M, K] w [N, K]^T, x rows xs elements apart. act 1 (silu), 2 (tanh gelu): out =
// act(x w[:N]^T) * (x w[N:]^T), w [2 N, K]. plan: oa_tile_gemm_plan's. scratch: splits * M * N floats,
// unused at one split; out null: left there, not added up.
extern "C" int oa_tile_gemm(void* stream, const void* x, int64_t xs, const void* w, void* out,
                            void* scratch, int M, int N, int K, int plan, int act) {
    const int form = plan >> 8, splits = plan & 255;
    if (M < 1 || N < 8 || N % 8 != 0 || K < 64 || K % 64 != 0) return -100;
    if (splits < 1 || splits > K / 64 || (splits > 1 ? !scratch || act : !out)) return -101;
    if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out | (uintptr_t)scratch) % 16 != 0 || xs % 8 != 0)
        return -102;
    if (act < 0 || act > 2 || plan < 0) return -104;
    if (xs < K || !tg_within(xs, N, K, act != 0)) return -103;
    const int rc = tg_run((hipStream_t)stream, x, xs * 2, w, nullptr, nullptr, out, splits > 1 ? scratch : nullptr,
                          M, N, (int64_t)K * 2, form, splits, act, false);
    return rc || splits == 1 || !out ? rc : oa_ring_sum(stream, scratch, out, M, N, splits);
}

// out [M, N] = (x8 [M, K] w8 [N, K]^T) * xscale[m] * wscale[n], e4m3 rows; form: oa_tile_gemm_fp8_form's
extern "C" int oa_tile_gemm_fp8(void* stream, const void* x8, const void* xscale, const void* w8,
                                const void* wscale, void* out, int M, int N, int K, int form) {
    if (M < 1 || N < 8 || N % 8 != 0 || K < 128 || K % 128 != 0 || K >= (1 << 23)) return -100;
    if (((uintptr_t)x8 | (uintptr_t)w8 | (uintptr_t)out) % 16 != 0) return -102;
    return tg_run((hipStream_t)stream, x8, K, w8, xscale, wscale, out, nullptr, M, N, K, form, 1, 0, true);
}

// out [M, N] = silu(gate) * up of the bf16 rows of such a product against w8 [2 N, K], gate rows first: a form of
// whole pairs of fragments (0 to 2)
extern "C" int oa_tile_gemm_fp8_silu(void* stream, const void* x8, const void* xscale, const void* w8,
                                     const void* wscale, void* out, int M, int N, int K, int form) {
    if (M < 1 || N < 8 || N % 8 != 0 || K < 128 || K % 128 != 0 || K >= (1 << 23)) return -100;
    if (((uintptr_t)x8 | (uintptr_t)w8 | (uintptr_t)out) % 16 != 0) return -102;
    // a lane's place in a strip of gate rows and their up rows is 32 bits wide
    if (((int64_t)N + 256) * K >= ((int64_t)1 << 32)) return -103;
    return tg_run((hipStream_t)stream, x8, K, w8, xscale, wscale, out, nullptr, M, N, K, form, 1, 1, true);
}
