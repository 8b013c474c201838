// Routed experts of prompt-sized batches on the matrix cores: five launches for
// a layer, static shapes, no host synchronisation (a per-expert loop of library
// products needs a device-to-host copy of the counts and about eight launches
// per used expert).
//
//   oa_moe_sort           pairs (token, choice) in expert order, expert offsets,
//                         the list of row tiles
//   oa_moe_grouped        MODE 1: mid[s] = act(gate) * up of the pair at sorted
//                         place s, its activation row gathered from x;
//                         MODE 2: mid[s] = relu(up)^2 (ungated experts);
//                         MODE 0: y[p] = pair_weight * (W2 mid[s]), scattered
//                         back to the pair's own row p
//   oa_moe_combine        out[t] = sum over a token's pairs, in their own order
//                         (+ another row, the shared expert's)
//
// A pair's result depends on no other pair, and a token's pairs are added in
// one order: the output does not depend on how pairs are placed in an expert.
// Activations are bf16; weights bf16, or fp8 (e4m3, one float32 scale per row)
// widened exactly to bf16 in registers. Sums are float32.
#include "skinny_strip.h"

typedef __attribute__((ext_vector_type(4))) unsigned int mgu4;
typedef __attribute__((ext_vector_type(8))) short mgs8;
typedef __attribute__((ext_vector_type(8))) __bf16 mgb8;
typedef __attribute__((ext_vector_type(2))) __bf16 mgb2;
typedef __attribute__((ext_vector_type(4))) float mgf4;

#define MG_MAX_E 1024

// ---- routing ----------------------------------------------------------------
// Router logits: float32 weights, products and sums on bf16 rows, on
// v_mfma_f32_16x16x4_f32. A block takes 16 experts, 16 tokens and one of `splits` parts
// of the columns, its four waves 16-column steps in turn, four steps' loads at a time;
// parts [splits, T, E] are added up in order by the choice below. Short loops on
// purpose: a step's other kernels leave neither the matrix nor this code in cache, and
// straight-line code that runs once waits for its own fetch. Us inside a step, both
// launches, 13 tokens x 64 experts x 2048: 9.9, 512 tokens 11.0 (22.2); before, logits and choice in one
// launch with a token per block, which drew the whole matrix through every block's CU:
// 20.9 (11.3 with it in cache), as unrolled vector code over the blocks 16.3.
__device__ __forceinline__ void moe_logits_part(const uint16_t* __restrict__ x, const float* __restrict__ rw,
                                                float* __restrict__ part, int T, int E, int K, int bt, int be,
                                                int bs, int splits, mgf4 (&red)[4][64]) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
    const int t0 = bt * 16, e0 = be * 16;
    const float* wr = rw + (size_t)min(e0 + r, E - 1) * K;
    const uint16_t* xr = x + (size_t)min(t0 + r, T - 1) * K;
    const int stride = splits * 64;     // columns between two steps of a wave
    mgf4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    // (blocks of more than four waves: the first four)
#pragma unroll 1
    for (int k0 = (bs * 4 + wid) * 16 + q * 4; k0 < K && wid < 4; k0 += 4 * stride) {
        mgf4 w[4];
        uint2 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {   // K % 4 == 0: a lane's four columns are all in or out
            const int k = min(k0 + i * stride, K - 4);
            w[i] = *reinterpret_cast<const mgf4*>(wr + k);
            v[i] = *reinterpret_cast<const uint2*>(xr + k);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool in = k0 + i * stride < K;
            const mgf4 f = {bf16_lo(v[i].x), bf16_hi(v[i].x), bf16_lo(v[i].y), bf16_hi(v[i].y)};
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? w[i][j] : 0.0f, in ? f[j] : 0.0f,
                                                           acc, 0, 0, 0);
        }
    }
    if (wid < 4) red[wid][lane] = acc;
    __syncthreads();
    if (wid) return;
    acc = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
    // D: column (token) lane & 15, rows (experts) (lane >> 4) * 4 and up
    if (t0 + r < T)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (e0 + q * 4 + j < E)
                part[((size_t)bs * T + t0 + r) * E + e0 + q * 4 + j] = acc[j];
}

__global__ __launch_bounds__(256) void moe_logits_kernel(const uint16_t* __restrict__ x,
                                                         const float* __restrict__ rw,
                                                         float* __restrict__ part, int T, int E,
                                                         int K) {
    __shared__ mgf4 red[4][64];
    moe_logits_part(x, rw, part, T, E, K, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.z, red);
}

// a op (a of the lane that DPP names); lanes without a source keep their value
template <int CTRL, typename F>
__device__ __forceinline__ int mg_dpp(int a, F op) {
    return op(a, __builtin_amdgcn_update_dpp(a, a, CTRL, 0xf, 0xf, false));
}
// over the wave by row shifts and row broadcasts: idempotent ops only
template <typename F>
__device__ __forceinline__ int mg_wave_all(int a, F op) {
    a = mg_dpp<0x111>(a, op);
    a = mg_dpp<0x112>(a, op);
    a = mg_dpp<0x114>(a, op);
    a = mg_dpp<0x118>(a, op);
    a = mg_dpp<0x142>(a, op);
    a = mg_dpp<0x143>(a, op);
    return __builtin_amdgcn_readlane(a, 63);
}
__device__ __forceinline__ float mg_wave_max(float v) {
    return __int_as_float(mg_wave_all(__float_as_int(v), [](int a, int b) {
        return __float_as_int(fmaxf(__int_as_float(a), __int_as_float(b)));
    }));
}

// Softmax and the `top` best experts, a wave per token; weights normalised over the
// chosen, ties go to the lower expert.
// z: E floats of the wave's own (a lane touches its own columns only). Lane r has the r-th choice and
// its weight.
__device__ __forceinline__ void moe_choose_token(const float* __restrict__ part, int t, int T, int E,
                                                 int top, int splits, float* z, int& who, float& weight) {
    const int lane = threadIdx.x & 63;
    float mx = -INFINITY;
    for (int e = lane; e < E; e += 64) {
        float a = 0.0f;
#pragma unroll 8
        for (int s = 0; s < splits; ++s) a += part[((size_t)s * T + t) * E + e];
        z[e] = a;
        mx = fmaxf(mx, a);
    }
    mx = mg_wave_max(mx);
    float sum = 0.0f;
    for (int e = lane; e < E; e += 64) sum += z[e] = expf(z[e] - mx);
    sum = wave_reduce_sum(sum);
    for (int e = lane; e < E; e += 64) z[e] = z[e] / sum;
    float mine = 0.0f, total = 0.0f;    // lane r keeps the r-th choice's score
    who = 0;
#pragma unroll 1
    for (int r = 0; r < top; ++r) {
        float bv = -INFINITY;
        int bi = 0x7fffffff;
        for (int e = lane; e < E; e += 64)
            if (z[e] > bv) {
                bv = z[e];
                bi = e;
            }
        const float best = mg_wave_max(bv);
        bi = mg_wave_all(bv == best ? bi : 0x7fffffff, [](int a, int b) { return min(a, b); });
        bv = best;
        if (bi == 0x7fffffff) {         // no score left that compares: a NaN or an infinite
            bi = 0;                     // logit makes all of a row NaN, and its weights too
            bv = NAN;
        }
        total += bv;
        if (lane == r) {
            mine = bv;
            who = bi;
        }
        if (lane == (bi & 63)) z[bi] = -INFINITY;   // the lane that reads it next
    }
    weight = mine / (total + 1e-20f);
}

__global__ __launch_bounds__(256) void moe_choose_kernel(const float* __restrict__ part,
                                                         int* __restrict__ idx,
                                                         float* __restrict__ wout,
                                                         int* __restrict__ tok, int T, int E,
                                                         int top, int splits) {
    __shared__ float zs[4][MG_MAX_E];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int t = blockIdx.x * 4 + wid;
    if (t >= T) return;
    int who;
    float weight;
    moe_choose_token(part, t, T, E, top, splits, zs[wid], who, weight);
    const size_t o = (size_t)t * top;
    if (lane < top) {
        idx[o + lane] = who;
        wout[o + lane] = weight;
        tok[o + lane] = t;
    }
}

// ---- sorting ----------------------------------------------------------------
// One block: counts per expert, offsets, tiles of `bm` rows, then the places.
// off [E + 1]; pre [E + 1]: first tile of every expert; tile_e: expert of every
// tile; perm [P]: pair at every sorted place.
// NT threads, no fewer than experts.
template <int NT, int MAXE>
struct SortRoom {
    int cnt[MAXE], cur[MAXE], wsum[2][NT / 64];
};
template <int NT, int MAXE>
__device__ __forceinline__ void moe_sort_pairs(const int* expert_ids, int P, int E, int bm,
                                               int* __restrict__ off, int* __restrict__ pre,
                                               int* __restrict__ tile_e, int* __restrict__ perm,
                                               SortRoom<NT, MAXE>& room) {
    auto &cnt = room.cnt, &cur = room.cur;
    auto& wsum = room.wsum;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    for (int e = tid; e < E; e += NT) cnt[e] = 0;
    __syncthreads();
    for (int p = tid; p < P; p += NT) {
        const int e = expert_ids[p];
        if ((unsigned)e < (unsigned)E) atomicAdd(&cnt[e], 1);
    }
    __syncthreads();
    // inclusive scans of rows and tiles, one expert per thread
    const int c = tid < E ? cnt[tid] : 0;
    const int nt = (c + bm - 1) / bm;
    int a = c, b = nt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int x = __shfl_up(a, o, 64), y = __shfl_up(b, o, 64);
        if (lane >= o) {
            a += x;
            b += y;
        }
    }
    if (lane == 63) {
        wsum[0][wid] = a;
        wsum[1][wid] = b;
    }
    __syncthreads();
    for (int w = 0; w < wid; ++w) {
        a += wsum[0][w];
        b += wsum[1][w];
    }
    if (tid < E) {
        off[tid + 1] = a;
        pre[tid + 1] = b;
        cur[tid] = a - c;
        for (int i = b - nt; i < b; ++i) tile_e[i] = tid;
    }
    if (tid == 0) off[0] = pre[0] = 0;
    __syncthreads();
    for (int p = tid; p < P; p += NT) {
        const int e = expert_ids[p];
        if ((unsigned)e < (unsigned)E) perm[atomicAdd(&cur[e], 1)] = p;
    }
}

__global__ __launch_bounds__(1024) void moe_sort_kernel(const int* __restrict__ expert_ids, int P,
                                                        int E, int bm, int* __restrict__ off,
                                                        int* __restrict__ pre,
                                                        int* __restrict__ tile_e,
                                                        int* __restrict__ perm) {
    __shared__ SortRoom<1024, MG_MAX_E> room;
    moe_sort_pairs(expert_ids, P, E, bm, off, pre, tile_e, perm, room);
}

// ---- routing beside the shared expert -------------------------------------------
// For a few tokens the routing is three launches on one to 64 blocks, one after the other, while the
// shared expert's two products could run: their strips (skinny.hip) and the logits share a launch,
// and so do the strips of the second product and one block that chooses and sorts for all tokens.
// The first blocks are the routing's. Each does what its own launch does, in the same order.
// Us inside a step, 64 experts of 1408 x 2048, top 6, a shared one of 2816, 13 tokens: five launches 29.2,
// two 17.6 (8.4 + 9.2: the second waits for its first block, two tokens a wave one after the other, the
// strips take 6.8). Code that runs once waits for its own fetch: with the logits of a wave's tokens
// asked for together, in straight lines, the second launch took 14.3. For more than 16 tokens one
// block is slow (four layers, 50 tokens 743 us, 785 with it), and with the sort apart nothing is won
// (24 tokens 941 / 928, 32 684 / 688).
#define MG_FRONT_E 256
#define MG_FRONT_T 16

template <int WV, int D>
__global__ __launch_bounds__(WV * 64) void moe_front_up_kernel(
    const uint16_t* __restrict__ x, const float* __restrict__ rw, float* __restrict__ part, int T, int E,
    int K, int splits, const uint16_t* __restrict__ w, uint16_t* __restrict__ mid, int I) {
    __shared__ __attribute__((aligned(16))) union {
        mgf4 logits[4][64];
        SkinnyRed<1, true, WV> strip;
    } room;
    const int te = CEIL_DIV(E, 16), logits = CEIL_DIV(T, 16) * te * splits;
    const int at = blockIdx.x;
    if (at < logits) moe_logits_part(x, rw, part, T, E, K, at / (te * splits), at / splits % te, at % splits, splits,
                                     room.logits);
    else skinny_strip<1, true, WV, D>(x, K, w, mid, T, I, K, 0, at - logits, room.strip);
}

// choice and sort of all tokens by one block of WV waves
template <int WV>
struct ChooseRoom {
    float z[WV][MG_FRONT_E];
    int ids[MG_FRONT_T * 64];
    SortRoom<WV * 64, MG_FRONT_E> sort;
};
template <int WV>
__device__ __forceinline__ void moe_choose_all(const float* __restrict__ part, int* __restrict__ idx,
                                               float* __restrict__ wout, int T, int E, int top, int splits,
                                               int bm, int* __restrict__ off, int* __restrict__ pre,
                                               int* __restrict__ tile_e, int* __restrict__ perm,
                                               ChooseRoom<WV>& room) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll 1
    for (int t = wid; t < T; t += WV) {
        int who;
        float weight;
        moe_choose_token(part, t, T, E, top, splits, room.z[wid], who, weight);
        if (lane < top) {
            room.ids[t * top + lane] = idx[t * top + lane] = who;
            wout[t * top + lane] = weight;
        }
    }
    __syncthreads();
    moe_sort_pairs(room.ids, T * top, E, bm, off, pre, tile_e, perm, room.sort);
}

__global__ __launch_bounds__(1024) void moe_choose_sort_kernel(
    const float* __restrict__ part, int* __restrict__ idx, float* __restrict__ wout, int T, int E, int top,
    int splits, int bm, int* __restrict__ off, int* __restrict__ pre, int* __restrict__ tile_e,
    int* __restrict__ perm) {
    __shared__ ChooseRoom<16> room;
    moe_choose_all(part, idx, wout, T, E, top, splits, bm, off, pre, tile_e, perm, room);
}

template <int WV, int D>
__global__ __launch_bounds__(WV * 64) void moe_front_down_kernel(
    const float* __restrict__ part, int* __restrict__ idx, float* __restrict__ wout, int T, int E, int top,
    int splits, int bm, int* __restrict__ off, int* __restrict__ pre, int* __restrict__ tile_e,
    int* __restrict__ perm, const uint16_t* __restrict__ mid, const uint16_t* __restrict__ w,
    uint16_t* __restrict__ out, int H, int I) {
    __shared__ __attribute__((aligned(16))) union {
        ChooseRoom<WV> choose;
        SkinnyRed<1, false, WV> strip;
    } room;
    if (blockIdx.x == 0) moe_choose_all(part, idx, wout, T, E, top, splits, bm, off, pre, tile_e, perm, room.choose);
    else skinny_strip<1, false, WV, D>(mid, I, w, out, T, H, I, 0, blockIdx.x - 1, room.strip);
}

// ---- grouped products ---------------------------------------------------------
__device__ __forceinline__ float mg_gate_act(float g, float u, int act, float limit, float alpha) {
    if (act == 2) {
        g = fminf(g, limit);
        u = fminf(fmaxf(u, -limit), limit);
        return g / (1.0f + __expf(-alpha * g)) * (u + 1.0f);
    }
    return g / (1.0f + __expf(-g)) * u;
}

// 8 fp8 (two words) to 8 bf16, exactly
__device__ __forceinline__ mgs8 mg_widen(uint32_t lo, uint32_t hi) {
    union {
        mgb2 h[4];
        mgs8 v;
    } r;
    r.h[0] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, false);
    r.h[1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, true);
    r.h[2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, false);
    r.h[3] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, true);
    return r.v;
}

template <int V>
__device__ __forceinline__ void mg_wait() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(V) : "memory");
}

// A block of four waves takes BM sorted rows of one expert and 128 of its weight rows (64
// gate and the 64 up rows beside them); a wave all rows by 32 of the strip, weights as the
// first operand of v_mfma_f32_16x16x32_bf16.
//
// What bounds it is the weight stream, up to some hundred rows an expert. Both operands come
// by 16-byte transfers straight into a ring of STAGES steps in LDS (a step: 128 bytes of every
// weight row and the same columns of the activation rows, whose addresses the lanes gather by
// expert), STAGES - 1 under way, two blocks a CU so that one streams while the other starts or
// ends. 16-byte chunk c of a 128-byte row r lies at c ^ (r >> 1 & 7), of a 256-byte one at c ^
// (r & 15): the rows of a fragment read touch every bank once. Weights of an expert with one
// row tile are read without being kept (nt), those of more tiles are met again in the die's L2.
// Work items are in an order that puts the row tiles of one expert and strip next to each
// other on ONE die (block ids go round the eight dies), and the dies share the items in use.
//
// Us over 2 GB of weights, up + down, with weight rows loaded one step ahead into registers
// (before) / here: 64 experts of 1408 x 2048, top 6, fp8: 13 tokens 63 + 36 / 47 + 27, 64
// tokens 78 + 47 / 57 + 32, 512 tokens 123 + 76 / 81 + 47; bf16: 8 tokens 92 + 56 / 65 + 32,
// 64 tokens 142 + 76 / 118 + 58, 512 tokens 201 + 111 / 134 + 72, 2048 tokens 317 + 192 /
// 233 + 158. The stream runs at 5.5 to 6.3 TB/s up to 6 rows an expert. One block a CU with
// six steps is slower (54 + 28 for 13 fp8 tokens), three with two are as fast (51 + 24).
// Strips that start apart, us, together / apart: 64 experts of 1408 x 2048, bf16: 13 tokens 94 +
// 45 / 91 + 45, 512 tokens 135 + 75 / 130 + 74, fp8 1500 tokens 193 + 106 / 167 + 104; 8 experts of
// 14336 x 4096, top 2, bf16: 13 tokens 292 + 164 / 276 + 139, 512 tokens 586 + 328 / 541 + 319.
template <int BM, int STAGES, bool FP8, int MODE>
__global__ __launch_bounds__(256, 2) void moe_grouped_kernel(
    const uint16_t* __restrict__ x, const char* __restrict__ w, const float* __restrict__ wscale,
    const int* __restrict__ off, const int* __restrict__ pre, const int* __restrict__ tile_e,
    const int* __restrict__ perm, const float* __restrict__ pair_w, uint16_t* __restrict__ out,
    int E, int N, int K, int top, int strips, int act, float limit, float alpha) {
    constexpr int FM = BM / 16;                  // activation fragments
    constexpr int XB = FP8 ? 256 : 128;          // bytes of an activation row in a step
    constexpr int XT = BM * XB / 1024;           // transfers of them; of a wave:
    constexpr int XPW = XT < 4 ? 1 : XT / 4;     // (two of 16 bf16 rows: waves repeat them)
    constexpr int LPS = 4 + XPW, STEP = 128 * 128 + BM * XB;
    extern __shared__ __attribute__((aligned(16))) char smem[];

    const int items = pre[E] * strips, per = (items + 7) >> 3;
    const int place = blockIdx.x >> 3, item = (blockIdx.x & 7) * per + place;
    if (place >= per || item >= items) return;
    const int e = tile_e[item / strips];
    const int t0 = pre[e], mt = pre[e + 1] - t0;
    const int in = item - t0 * strips;
    const int strip = in / mt, mtile = in - strip * mt;
    const int s0 = off[e] + mtile * BM;
    const int m = min(BM, off[e + 1] - s0);
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t rb = FP8 ? (int64_t)K : 2 * (int64_t)K;    // bytes of a weight row
    const int ns = (int)(rb / 128);

    // Strips start at steps of their own, the row tiles of one together: rows a few KiB apart
    // lie on the same memory channels, and blocks that read the same columns share those. Narrow
    // fp8 tiles lose more by it (64 x 1408 x 2048, 13 tokens 47.5 us, 48.2) than they win.
    constexpr bool TURN = !FP8 || BM >= 64;
    const int turned = TURN ? (e * strips + strip) * 3 % ns : 0;
    int ahead = ns - turned;                         // steps to the last column

    // this lane's row and chunk of every transfer; weight rows past N repeat the last one,
    // rows past the end of the expert's too
    const char* src[LPS];
    uint32_t dst[LPS];
    const char* we = w + (int64_t)e * (MODE == 1 ? 2 * N : N) * rb;
    const uint32_t base = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem);
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const int row = (wid * 4 + p) * 8 + (lane >> 3);
        int64_t at;
        if (MODE == 1) at = min(strip * 64 + (row >> 5) * 16 + (row & 15), N - 1) + (row & 16 ? N : 0);
        else at = min(strip * 128 + row, N - 1);
        src[p] = we + at * rb + turned * 128 + ((lane & 7) ^ (row >> 1 & 7)) * 16;
        dst[p] = base + (wid * 4 + p) * 1024;
    }
#pragma unroll
    for (int p = 0; p < XPW; ++p) {
        const int tr = XT < 4 ? wid % XT : p * 4 + wid;
        const int row = tr * (1024 / XB) + lane / (XB / 16);
        const int chunk = FP8 ? (lane & 15) ^ (row & 15) : (lane & 7) ^ (row >> 1 & 7);
        const int s = s0 + min(row, m - 1);
        src[4 + p] = reinterpret_cast<const char*>(x) +
                     (int64_t)(MODE == 0 ? s : perm[s] / top) * K * 2 + turned * XB + chunk * 16;
        dst[4 + p] = base + 128 * 128 + tr * 1024;
    }
    auto stage = [&](int buf) {
#pragma unroll
        for (int p = 0; p < LPS; ++p) {
            if (p < 4 && mt == 1) lds_transfer16<true>(dst[p] + buf * STEP, src[p]);
            else lds_transfer16(dst[p] + buf * STEP, src[p]);
            src[p] += p < 4 ? 128 : XB;
        }
        if (TURN && --ahead == 0) {
#pragma unroll
            for (int p = 0; p < LPS; ++p) src[p] -= ns * (p < 4 ? 128 : XB);
        }
    };

    mgf4 acc[2][FM] = {};
#pragma unroll
    for (int t = 0; t < STAGES - 1; ++t)
        if (t < ns) stage(t);
    int buf = 0;
    for (int t = 0; t < ns; ++t) {
        const int behind = min(STAGES - 2, ns - 1 - t);      // younger steps under way
        if (STAGES > 3 && behind >= 2) mg_wait<2 * LPS>();
        else if (STAGES > 2 && behind >= 1) mg_wait<LPS>();
        else mg_wait<0>();
        if (t + STAGES - 1 < ns) stage(buf == 0 ? STAGES - 1 : buf - 1);
        const char* bx = smem + buf * STEP + 128 * 128;
        const char* bw = smem + buf * STEP + wid * 32 * 128;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int at = r * 128 + (((h * 4 + q) ^ (r >> 1)) << 4);
            mgu4 v[2];
#pragma unroll
            for (int f = 0; f < 2; ++f) v[f] = *reinterpret_cast<const mgu4*>(bw + f * 16 * 128 + at);
            // fp8: 16 bytes hold the lane's columns of two products
#pragma unroll
            for (int k = 0; k < (FP8 ? 2 : 1); ++k) {
                mgs8 a[2];
#pragma unroll
                for (int f = 0; f < 2; ++f)
                    a[f] = !FP8 ? __builtin_bit_cast(mgs8, v[f])
                           : k  ? mg_widen(v[f][2], v[f][3])
                                : mg_widen(v[f][0], v[f][1]);
#pragma unroll
                for (int j = 0; j < FM; ++j) {
                    const mgs8 b = *reinterpret_cast<const mgs8*>(
                        bx + (FP8 ? (j * 16 + r) * 256 + (((h * 8 + q * 2 + k) ^ r) << 4)
                                  : j * 16 * 128 + at));
#pragma unroll
                    for (int f = 0; f < 2; ++f)
                        acc[f][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(mgb8, a[f]), __builtin_bit_cast(mgb8, b), acc[f][j], 0, 0, 0);
                }
            }
        }
        buf = buf + 1 == STAGES ? 0 : buf + 1;
    }

    // lane: sorted row r of a fragment, weight rows q * 4 .. + 3
    const int n0 = MODE == 1 ? strip * 64 + wid * 16 : strip * 128 + wid * 32;
    float sc[2][4];
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (!FP8) {
                sc[f][i] = 1.0f;
                continue;
            }
            const int n = min(n0 + (MODE == 1 ? 0 : f * 16) + q * 4 + i, N - 1);
            sc[f][i] = wscale[(size_t)e * (MODE == 1 ? 2 * N : N) + (MODE == 1 && f ? N + n : n)];
        }
#pragma unroll
    for (int j = 0; j < FM; ++j) {
        const int row = j * 16 + r;
        if (row >= m) continue;
        if (MODE == 1) {
            uint32_t o[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float v0 = mg_gate_act(acc[0][j][2 * h] * sc[0][2 * h],
                                             acc[1][j][2 * h] * sc[1][2 * h], act, limit, alpha);
                const float v1 = mg_gate_act(acc[0][j][2 * h + 1] * sc[0][2 * h + 1],
                                             acc[1][j][2 * h + 1] * sc[1][2 * h + 1], act, limit, alpha);
                o[h] = pack_bf16x2(v0, v1);
            }
            *reinterpret_cast<uint2*>(out + (size_t)(s0 + row) * N + n0 + q * 4) = make_uint2(o[0], o[1]);
        } else {
            const int pair = MODE == 0 ? perm[s0 + row] : 0;
            const float pw = MODE == 0 ? pair_w[pair] : 1.0f;
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                const int n = n0 + f * 16 + q * 4;
                if (n >= N) continue;              // N is a multiple of 16
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v[i] = acc[f][j][i] * sc[f][i];
                    if (MODE == 2) {
                        v[i] = fmaxf(v[i], 0.0f);
                        v[i] *= v[i];
                    } else {
                        v[i] *= pw;
                    }
                }
                *reinterpret_cast<uint2*>(out + (size_t)(MODE == 0 ? pair : s0 + row) * N + n) =
                    make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
            }
        }
    }
}

// ---- sum over a token's pairs ---------------------------------------------------
// eight channels per thread; `more` (optional) is added as one more row
__global__ __launch_bounds__(256) void moe_combine_kernel(const uint16_t* __restrict__ y,
                                                          const uint16_t* __restrict__ more,
                                                          uint16_t* __restrict__ out, int top,
                                                          int H8, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const int64_t t = i / H8, c = i - t * H8;
        const uint4* yr = reinterpret_cast<const uint4*>(y) + t * top * H8 + c;
        float s[8] = {};
        for (int k = 0; k < top; ++k) {
            const uint4 v = yr[(int64_t)k * H8];
            const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                s[2 * j] += bf16_lo(u[j]);
                s[2 * j + 1] += bf16_hi(u[j]);
            }
        }
        if (more) {
            const uint4 v = reinterpret_cast<const uint4*>(more)[i];
            const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                s[2 * j] += bf16_lo(u[j]);
                s[2 * j + 1] += bf16_hi(u[j]);
            }
        }
        reinterpret_cast<uint4*>(out)[i] = make_uint4(pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3]),
                                                      pack_bf16x2(s[4], s[5]), pack_bf16x2(s[6], s[7]));
    }
}

// Parts of the columns: enough blocks for the chip, no fewer than four steps a wave.
static int moe_route_splits(int T, int E, int K) {
    const int64_t tiles = (int64_t)CEIL_DIV(T, 16) * CEIL_DIV(E, 16);
    return (int)max((int64_t)1, min(min((int64_t)16, 1024 / tiles), (int64_t)CEIL_DIV(K, 256)));
}

// floats of oa_moe_route's scratch
extern "C" int64_t oa_moe_route_scratch(int T, int E, int K) {
    return (int64_t)moe_route_splits(T, E, K) * T * E;
}

// idx, w, tok [T, top]: expert, weight and token of every pair
extern "C" int oa_moe_route(void* stream, const void* x, const void* rw, void* scratch, void* idx,
                            void* w, void* tok, int T, int E, int K, int top) {
    if (T < 1 || E < 1 || E > MG_MAX_E || top < 1 || top > E || top > 64 || K < 4 || K % 4 != 0)
        return -100;
    const int splits = moe_route_splits(T, E, K);
    hipLaunchKernelGGL(moe_logits_kernel, dim3(CEIL_DIV(T, 16), CEIL_DIV(E, 16), splits), dim3(256),
                       0, (hipStream_t)stream, (const uint16_t*)x, (const float*)rw,
                       (float*)scratch, T, E, K);
    hipLaunchKernelGGL(moe_choose_kernel, dim3(CEIL_DIV(T, 4)), dim3(256), 0, (hipStream_t)stream,
                       (const float*)scratch, (int*)idx, (float*)w, (int*)tok, T, E, top, splits);
    HIP_CHECK_LAUNCH();
    return 0;
}

// Router logits' parts into scratch (oa_moe_route_scratch) and, with gate_up [2I, K], beside them
// mid [T, I] = silu(x gate^T) * (x up^T): two of the four steps of a layer's routing and shared expert.
extern "C" int oa_moe_front_up(void* stream, const void* x, const void* rw, void* scratch, int T, int E, int K,
                               const void* gate_up, void* mid, int I) {
    if (T < 1 || E < 1 || E > MG_MAX_E || K < 4 || K % 4 != 0) return -100;
    const int splits = moe_route_splits(T, E, K);
    const int logits = CEIL_DIV(T, 16) * CEIL_DIV(E, 16) * splits;
    hipStream_t st = (hipStream_t)stream;
    if (!gate_up) {
        hipLaunchKernelGGL(moe_logits_kernel, dim3(CEIL_DIV(T, 16), CEIL_DIV(E, 16), splits), dim3(256), 0, st,
                           (const uint16_t*)x, (const float*)rw, (float*)scratch, T, E, K);
        HIP_CHECK_LAUNCH();
        return 0;
    }
    if (T > MG_FRONT_T || I < 1 || K < 32 || K % 32 != 0) return -101;
#define MFU(WV)                                                                                        \
    hipLaunchKernelGGL((moe_front_up_kernel<WV, 8>), dim3(logits + CEIL_DIV(I, 16)), dim3((WV) * 64), 0, \
                       st, (const uint16_t*)x, (const float*)rw, (float*)scratch, T, E, K, splits,     \
                       (const uint16_t*)gate_up, (uint16_t*)mid, I)
    // the forms of oa_skinny
    if (K <= 2048) MFU(4);
    else MFU(8);
#undef MFU
    HIP_CHECK_LAUNCH();
    return 0;
}

// Choice and sort from the logits' parts (idx, w [T, top], lists as of oa_moe_sort) and, with down
// [H, I], beside them out [T, H] = mid down^T.
extern "C" int oa_moe_front_down(void* stream, const void* scratch, void* idx, void* w, int T, int E, int K,
                                 int top, int bm, void* off, void* pre, void* tile_e, void* perm,
                                 const void* mid, const void* down, void* out, int H, int I) {
    if (T < 1 || T > MG_FRONT_T || E < 1 || E > MG_FRONT_E || top < 1 || top > E || top > 64 ||
        (bm != 16 && bm != 32 && bm != 64 && bm != 128))
        return -100;
    const int splits = moe_route_splits(T, E, K);
    hipStream_t st = (hipStream_t)stream;
    if (!down) {
        hipLaunchKernelGGL(moe_choose_sort_kernel, dim3(1), dim3(1024), 0, st, (const float*)scratch, (int*)idx,
                           (float*)w, T, E, top, splits, bm, (int*)off, (int*)pre, (int*)tile_e, (int*)perm);
        HIP_CHECK_LAUNCH();
        return 0;
    }
    if (H < 1 || I < 32 || I % 32 != 0) return -101;
#define MFD(WV)                                                                                          \
    hipLaunchKernelGGL((moe_front_down_kernel<WV, 8>), dim3(1 + CEIL_DIV(H, 16)), dim3((WV) * 64), 0, st, \
                       (const float*)scratch, (int*)idx, (float*)w, T, E, top, splits, bm, (int*)off,    \
                       (int*)pre, (int*)tile_e, (int*)perm, (const uint16_t*)mid, (const uint16_t*)down, \
                       (uint16_t*)out, H, I)
    if (I >= 2 * H) MFD(4);
    else MFD(8);
#undef MFD
    HIP_CHECK_LAUNCH();
    return 0;
}

extern "C" int oa_moe_sort(void* stream, const void* expert_ids, int P, int E, int bm, void* off,
                           void* pre, void* tile_e, void* perm) {
    if (P < 1 || E < 1 || E > MG_MAX_E || (bm != 16 && bm != 32 && bm != 64 && bm != 128)) return -100;
    hipLaunchKernelGGL(moe_sort_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream,
                       (const int*)expert_ids, P, E, bm, (int*)off, (int*)pre, (int*)tile_e, (int*)perm);
    HIP_CHECK_LAUNCH();
    return 0;
}

// mode 0: x = mid [P, K], w [E, N, K], out = y [P, N]; mode 1: x [T, K],
// w [E, 2N, K], out = mid [P, N]; mode 2: x [T, K], w [E, N, K], out = mid.
// max_tiles: no fewer than the tiles that oa_moe_sort can make of P pairs.
extern "C" int oa_moe_grouped(void* stream, const void* x, const void* w, const void* wscale,
                              const void* off, const void* pre, const void* tile_e, const void* perm,
                              const void* pair_w, void* out, int E, int N, int K, int top, int bm,
                              int max_tiles, int mode, int act, float limit, float alpha) {
    if (K < 128 || K % 128 != 0 || N < 16 || N % 16 != 0 || (mode == 1 && N % 64 != 0) || top < 1 ||
        max_tiles < 1 || E < 1 || mode < 0 || mode > 2)
        return -100;
    const int strips = mode == 1 ? N / 64 : CEIL_DIV(N, 128);
    const int64_t items = (int64_t)strips * max_tiles;
    if (items > (1 << 28)) return -101;
    const dim3 grid((unsigned)(CEIL_DIV(items, 8) * 8)), block(256);
#define MG(BMV, ST, F, MO)                                                                         \
    hipLaunchKernelGGL((moe_grouped_kernel<BMV, ST, F, MO>), grid, block,                          \
                       (ST) * (128 * 128 + (BMV) * ((F) ? 256 : 128)), (hipStream_t)stream,        \
                       (const uint16_t*)x, (const char*)w, (const float*)wscale, (const int*)off,  \
                       (const int*)pre, (const int*)tile_e, (const int*)perm, (const float*)pair_w, \
                       (uint16_t*)out, E, N, K, top, strips, act, limit, alpha)
#define MGM(BMV, ST, F)                    \
    do {                                   \
        if (mode == 0) MG(BMV, ST, F, 0);  \
        else if (mode == 1) MG(BMV, ST, F, 1); \
        else MG(BMV, ST, F, 2);            \
    } while (0)
    // steps: as many as two blocks' rings leave room for
    switch (bm + (wscale ? 1 : 0)) {
        case 16: MGM(16, 4, false); break;
        case 17: MGM(16, 4, true); break;
        case 32: MGM(32, 4, false); break;
        case 33: MGM(32, 3, true); break;
        case 64: MGM(64, 3, false); break;
        case 65: MGM(64, 2, true); break;
        case 128: MGM(128, 2, false); break;
        default: return -102;
    }
#undef MGM
#undef MG
    HIP_CHECK_LAUNCH();
    return 0;
}

extern "C" int oa_moe_combine(void* stream, const void* y, const void* more, void* out, int T,
                              int top, int H) {
    if (T < 1 || top < 1 || H < 8 || H % 8 != 0) return -100;
    const int64_t n = (int64_t)T * (H / 8);
    const int64_t blocks = CEIL_DIV(n, 256);
    hipLaunchKernelGGL(moe_combine_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0,
                       (hipStream_t)stream, (const uint16_t*)y, (const uint16_t*)more, (uint16_t*)out,
                       top, H / 8, n);
    HIP_CHECK_LAUNCH();
    return 0;
}
