// Fused grammar-mask + greedy sampling kernel.
//
// Constrained JSON and tool calls: replaces the reference's post-hoc JSON
// repair (pkg/utils/json.go:16-190) by making invalid JSON impossible. The FSM advances on the CPU (C++ — grammar_fsm.cpp); each step
// it produces a per-sequence allowed-token BITMASK (V/32 words, ~16 KB for a
// 128k vocab) which this kernel fuses with the argmax over the logits row —
// one read of the logits, no [B, V] masked-softmax intermediate.
//
// logits bf16 [B, V]; mask uint32 [B, ceil(V/32)] (bit t set = allowed;
// nullptr -> unconstrained); out int32 [B], -1 where nothing is allowed.

#include "common.h"

__device__ __forceinline__ uint32_t ordered_f32(float f) {
    union {
        uint32_t u;
        float f;
    } v;
    v.f = f;
    return (v.u & 0x80000000u) ? ~v.u : (v.u | 0x80000000u);
}

// One block of 16 waves per row, one launch: in a chain of small kernels a launch costs
// more than a CU needs for a row, 256 KB at 128k tokens, with 8 loads of 16 bytes a lane
// under way (16 blocks a row with an atomic maximum, a fill before and a launch after:
// 11.6 us of a decode step of one row of 32000; here 5.8). A lane keeps its best group of 8
// tokens, a comparison and a selection a token, and only the row's best group is looked
// through for the token. Lowest index wins ties (-0 and +0 are one); NaN and -inf are never
// chosen. The instruction for a maximum would take half as many (back to back, one row of
// 32000 with a mask 5.2 us beside 5.6, of 128256 without 4.9 beside 6.0), but answers a
// signaling NaN with NaN and so loses the tokens before it.
template <bool MASK>
__global__ __launch_bounds__(1024) void masked_argmax_kernel(
    const uint4* __restrict__ logits, const uint32_t* __restrict__ mask, int* __restrict__ out,
    int groups, int mask_words) {
    const int b = blockIdx.x, lane = threadIdx.x & (WAVE - 1), wid = threadIdx.x / WAVE;
    const uint4* row = logits + (size_t)b * groups;
    const uint8_t* mrow = MASK ? (const uint8_t*)(mask + (size_t)b * mask_words) : nullptr;
    constexpr int N = 8;
    float best = -INFINITY;
    int at = groups;
    for (int i0 = threadIdx.x; i0 < groups; i0 += 1024 * N) {
        uint4 w[N];
        uint32_t allow[N];
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const int i = min(i0 + 1024 * u, groups - 1);      // a repeat is never better
            w[u] = row[i];
            allow[u] = MASK ? mrow[i] : 0xffu;
        }
#pragma unroll
        for (int u = 0; u < N; ++u) {
            float m = -INFINITY;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float lo = bf16_lo((&w[u].x)[j]), hi = bf16_hi((&w[u].x)[j]);
                m = (!MASK || (allow[u] >> (2 * j) & 1)) && lo > m ? lo : m;
                m = (!MASK || (allow[u] >> (2 * j + 1) & 1)) && hi > m ? hi : m;
            }
            if (m > best) {
                best = m;
                at = min(i0 + 1024 * u, groups - 1);
            }
        }
    }
    __shared__ float sv[16];
    __shared__ int si[16];
    auto take = [&](float v, int i) {
        if (v > best || (v == best && i < at)) {
            best = v;
            at = i;
        }
    };
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        take(__shfl_xor(best, off, WAVE), __shfl_xor(at, off, WAVE));
    if (lane == 0) {
        sv[wid] = best;
        si[wid] = at;
    }
    __syncthreads();
    if (wid > 0) return;
    best = sv[lane & 15];
    at = si[lane & 15];
#pragma unroll
    for (int off = 8; off > 0; off >>= 1)
        take(__shfl_xor(best, off, WAVE), __shfl_xor(at, off, WAVE));
    if (lane > 0) return;
    int tok = -1;
    if (at < groups) {
        const uint4 w = row[at];
        const uint32_t allow = MASK ? mrow[at] : 0xffu;
#pragma unroll
        for (int j = 7; j >= 0; --j) {
            const uint32_t x = (&w.x)[j / 2];
            if ((allow >> j & 1) && (j % 2 ? bf16_hi(x) : bf16_lo(x)) == best) tok = at * 8 + j;
        }
    }
    out[b] = tok;
}

extern "C" int oa_masked_argmax(void* stream, const void* logits, const void* mask, void* out,
                                int B, int V) {
    if (V % 8 != 0) return -100;
    if (B <= 0) return 0;
    auto kernel = mask ? masked_argmax_kernel<true> : masked_argmax_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3(B), dim3(1024), 0, (hipStream_t)stream, (const uint4*)logits,
                       (const uint32_t*)mask, (int*)out, V / 8, CEIL_DIV(V, 32));
    HIP_CHECK_LAUNCH();
    return 0;
}

// float32 logits (models whose head emits float32, any V): grid (chunks, B);
// each block scans its part of the row and leaves its best (value, index)
// in ws[b][chunk]; a second small kernel picks among the chunks. Lowest
// index wins ties, -1 if nothing is allowed. No atomics, nothing to clear.
#define F32_CHUNKS 16
__device__ __forceinline__ bool better_f32(float v, int i, float bv, int bi) {
    return i >= 0 && (bi < 0 || v > bv || (v == bv && i < bi));
}

__global__ __launch_bounds__(256) void masked_argmax_f32_scan(
    const float* __restrict__ logits, const uint32_t* __restrict__ mask,
    float* __restrict__ ws_val, int* __restrict__ ws_idx, int V, int mask_words) {
    const int b = blockIdx.y, chunk = blockIdx.x;
    const float* row = logits + (size_t)b * V;
    const uint32_t* mrow = mask ? mask + (size_t)b * mask_words : nullptr;
    const int per = CEIL_DIV(V, F32_CHUNKS);
    const int t0 = chunk * per, t1 = min(V, t0 + per);
    float best = -INFINITY;
    int besti = -1;
    for (int t = t0 + threadIdx.x; t < t1; t += blockDim.x) {
        if (mrow && !((mrow[t >> 5] >> (t & 31)) & 1u)) continue;
        const float v = row[t];
        if (besti < 0 || v > best) {  // ascending t per thread: first max kept
            best = v;
            besti = t;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(best, off, WAVE);
        const int oi = __shfl_xor(besti, off, WAVE);
        if (better_f32(ov, oi, best, besti)) {
            best = ov;
            besti = oi;
        }
    }
    __shared__ float sv[4];
    __shared__ int si[4];
    const int wid = threadIdx.x / WAVE;
    if ((threadIdx.x & (WAVE - 1)) == 0) {
        sv[wid] = best;
        si[wid] = besti;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w)
            if (better_f32(sv[w], si[w], best, besti)) {
                best = sv[w];
                besti = si[w];
            }
        ws_val[b * F32_CHUNKS + chunk] = best;
        ws_idx[b * F32_CHUNKS + chunk] = besti;
    }
}

__global__ void masked_argmax_f32_finish(const float* __restrict__ ws_val,
                                         const int* __restrict__ ws_idx,
                                         int* __restrict__ out, int B) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    float best = -INFINITY;
    int besti = -1;
    for (int c = 0; c < F32_CHUNKS; ++c)
        if (better_f32(ws_val[b * F32_CHUNKS + c], ws_idx[b * F32_CHUNKS + c], best, besti)) {
            best = ws_val[b * F32_CHUNKS + c];
            besti = ws_idx[b * F32_CHUNKS + c];
        }
    out[b] = besti;
}

// ws: B * F32_CHUNKS * 8 bytes of scratch
extern "C" int oa_masked_argmax_f32(void* stream, const void* logits, const void* mask,
                                    void* ws, void* out, int B, int V) {
    if (B <= 0) return 0;
    float* ws_val = (float*)ws;
    int* ws_idx = (int*)ws + (size_t)B * F32_CHUNKS;
    hipLaunchKernelGGL(masked_argmax_f32_scan, dim3(F32_CHUNKS, B), dim3(256), 0,
                       (hipStream_t)stream, (const float*)logits, (const uint32_t*)mask,
                       ws_val, ws_idx, V, CEIL_DIV(V, 32));
    HIP_CHECK_LAUNCH();
    hipLaunchKernelGGL(masked_argmax_f32_finish, dim3(CEIL_DIV(B, 64)), dim3(64), 0,
                       (hipStream_t)stream, (const float*)ws_val, (const int*)ws_idx,
                       (int*)out, B);
    HIP_CHECK_LAUNCH();
    return 0;
}

// Log-probability of a chosen token and the most likely tokens of a row, for B rows of
// float32 or bf16 logits. Two launches and nothing of the row's size written: a wave takes
// 1024 logits in registers and leaves their maximum, the sum of exponentials under it and
// its `top` best; a block per row merges those. What bounds it is the two launches: one row
// of 128256 bf16 takes 12.5 us with its 5 best (5.6 with none, 46 with 20), where a float32 copy, log-softmax, a sort of the row and
// the lookups took 150 and the host waited for each of them.
//
// An entry is value << 32 | ~index in an order that floats keep as integers: equal values go
// by index (-0 and +0 are one), NaN is the largest. Every entry lies above 0 and below
// LP_START, also a NaN's at index 0: a merge that takes the largest below the last one finds
// all that are there.
typedef unsigned long long lp_u64;
#define LP_START (~(lp_u64)0)

__device__ __forceinline__ float lp_load(const float* p) { return *p; }
__device__ __forceinline__ float lp_load(const uint16_t* p) { return bf16_to_f32(*p); }

__device__ __forceinline__ lp_u64 lp_entry(float v, int i) {
    const uint32_t key = v != v ? 0xfffffffeu : ordered_f32(v + 0.0f);    // -0 + 0 is +0
    return (lp_u64)key << 32 | (uint32_t)~i;
}
__device__ __forceinline__ lp_u64 wave_max_u64(lp_u64 v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const lp_u64 o = __shfl_xor(v, off, WAVE);
        v = o > v ? o : v;
    }
    return v;
}

// best [B, waves, top], ms [B, waves, 2]
template <typename T>
__global__ __launch_bounds__(256) void logprob_scan_kernel(const T* __restrict__ logits, int64_t stride,
                                                           lp_u64* __restrict__ best,
                                                           float* __restrict__ ms, int V, int waves,
                                                           int top) {
    const int lane = threadIdx.x & 63, wave = blockIdx.x * 4 + (threadIdx.x >> 6), b = blockIdx.y;
    if (wave >= waves) return;
    const T* row = logits + b * stride;
    float v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int t = wave * 1024 + i * 64 + lane;
        v[i] = lp_load(row + min(t, V - 1));
        if (t >= V) v[i] = -INFINITY;
    }
    float m = v[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) m = fmaxf(m, v[i]);
    m = wave_reduce_max(m);
    const float ref = m == -INFINITY ? 0.0f : m;
    float s = 0.0f;
    lp_u64 e[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int t = wave * 1024 + i * 64 + lane;
        s += expf(v[i] - ref);
        e[i] = t < V ? lp_entry(v[i], t) : 0;
    }
    s = wave_reduce_sum(s);
    const int64_t at = (int64_t)b * waves + wave;
    if (lane == 0) {
        ms[at * 2] = m;
        ms[at * 2 + 1] = s;
    }
    for (int r = 0; r < top; ++r) {
        lp_u64 x = e[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) x = e[i] > x ? e[i] : x;
        x = wave_max_u64(x);
        if (lane == 0) best[at * top + r] = x;
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (e[i] == x) e[i] = 0;
    }
}

// out [B, 1 + 2 * top]: log-probability of tokens[b] (NaN where it is no token), then index
// and log-probability of the best
template <typename T>
__global__ __launch_bounds__(256) void logprob_finish_kernel(
    const T* __restrict__ logits, int64_t stride, const int* __restrict__ tokens,
    const lp_u64* __restrict__ best, const float* __restrict__ ms, int* __restrict__ out, int V,
    int waves, int top) {
    __shared__ float red[4];
    __shared__ lp_u64 win[4];
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    ms += (int64_t)b * waves * 2;
    best += (int64_t)b * waves * top;
    out += (int64_t)b * (1 + 2 * top);
    float m = -INFINITY;
    for (int w = tid; w < waves; w += 256) m = fmaxf(m, ms[w * 2]);
    m = wave_reduce_max(m);
    if (lane == 0) red[wid] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    __syncthreads();
    // a part without a finite logit has the sum zero; a NaN in any part is in its sum
    float s = 0.0f;
    for (int w = tid; w < waves; w += 256) s += ms[w * 2 + 1] * expf(ms[w * 2] - m);
    s = wave_reduce_sum(s);
    if (lane == 0) red[wid] = s;
    __syncthreads();
    const float ls = logf((red[0] + red[1]) + (red[2] + red[3]));
    const T* row = logits + b * stride;
    if (tid == 0) {
        const int t = tokens[b];
        out[0] = __float_as_int(t >= 0 && t < V ? (lp_load(row + t) - m) - ls : NAN);
    }
    lp_u64 prev = LP_START;
    for (int r = 0; r < top; ++r) {
        lp_u64 x = 0;
        for (int i = tid; i < waves * top; i += 256) {
            const lp_u64 c = best[i];
            if (c < prev && c > x) x = c;
        }
        x = wave_max_u64(x);
        if (lane == 0) win[wid] = x;
        __syncthreads();
        x = max(max(win[0], win[1]), max(win[2], win[3]));
        prev = x;
        if (tid == 0) {
            const int t = (int)~(uint32_t)x;         // found: top <= V, and no wave has less to give
            out[1 + 2 * r] = t;
            out[2 + 2 * r] = __float_as_int((lp_load(row + t) - m) - ls);
        }
        __syncthreads();
    }
}

// rows `stride` elements apart; top at most 32 and V. ws: B * ceil(V / 1024) * (top + 1) * 8
// bytes, 8-byte aligned.
extern "C" int oa_token_logprobs(void* stream, const void* logits, int64_t stride, const void* tokens,
                                 void* ws, void* out, int B, int V, int top, int is_f32) {
    if (B < 1 || V < 1 || top < 0 || top > 32 || top > V || B > 65535) return -100;
    const int waves = CEIL_DIV(V, 1024);
    lp_u64* best = (lp_u64*)ws;
    float* ms = (float*)(best + (int64_t)B * waves * top);
    const dim3 grid(CEIL_DIV(waves, 4), B);
    hipStream_t s = (hipStream_t)stream;
#define LP(T)                                                                                       \
    do {                                                                                            \
        hipLaunchKernelGGL((logprob_scan_kernel<T>), grid, dim3(256), 0, s, (const T*)logits, stride, \
                           best, ms, V, waves, top);                                                 \
        HIP_CHECK_LAUNCH();                                                                         \
        hipLaunchKernelGGL((logprob_finish_kernel<T>), dim3(B), dim3(256), 0, s, (const T*)logits,   \
                           stride, (const int*)tokens, best, ms, (int*)out, V, waves, top);          \
        HIP_CHECK_LAUNCH();                                                                         \
    } while (0)
    if (is_f32) LP(float);
    else LP(uint16_t);
#undef LP
    return 0;
}
