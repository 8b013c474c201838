// Skinny-M GEMM ("GEMV") for decode projections on MI355X:
//   out[M, N] = x[M, K] @ W[N, K]^T      (torch F.linear layout, bf16)
//
// Decode at small batch is weight-streaming-bound: each step reads every
// weight byte once. hipBLASLt's skinny kernels measure ~2.5x off the HBM
// roofline at M=1 (19.9us for a 50 MB qkv read, ~8us at 6.3 TB/s); this
// kernel follows the CDNA guide's GEMV row ("M <= 16 decode weights: operand
// streamed once per block, not shared across waves -> load straight to
// VGPRs, deep unroll, late vmcnt"): W rows stream through 16-B vector loads
// per lane, fp32 accumulate, one wave-reduction per (row, m). The activation
// x is tiny (8-56 KB) and L1-resident after the first pass — each lane
// re-reads only its own 16-B slices, so no LDS staging is needed.
//
// Requires K % 512 == 0 (64 lanes x 8 bf16); callers fall back to hipBLASLt
// otherwise (and for M > 8, where the MFMA path wins).

#include <type_traits>

#include "mixer_util.h"

typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

__device__ __forceinline__ u32x4 nt_load4(const uint32_t* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}


// fp32 rstd of x row m: one extra pass over the (L1-resident) activation
__device__ __forceinline__ float row_rstd(const uint32_t* xrow, int k2, int lane,
                                          float eps) {
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

// NORM: x is normalized on the fly (rstd prologue + norm-weight multiply) —
// the separate rmsnorm kernel and its output round-trip disappear.
// ADDRES: the epilogue adds a residual row — out = x @ W^T + residual, i.e.
// the new residual stream is produced directly by the projection.
template <int M, bool NORM, bool ADDRES, int RW = 2>
__global__ __launch_bounds__(256) void gemv_kernel(
    const uint32_t* __restrict__ x,  // [M, K/2]
    const uint32_t* __restrict__ w,  // [N, K/2]
    uint32_t* __restrict__ out,      // [M, N] bf16 (u16 scalar writes)
    const uint32_t* __restrict__ wn, // [K/2] rmsnorm weight (NORM only)
    const uint32_t* __restrict__ res,// [M, N] residual (ADDRES only)
    int N, int k2 /* K/2 */, float eps) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int wid = threadIdx.x / WAVE;

    float rstd[M];
    if (NORM) {
#pragma unroll
        for (int m = 0; m < M; ++m) rstd[m] = row_rstd(x + (size_t)m * k2, k2, lane, eps);
    }

    // RW adjacent W rows per wave: multiplies the outstanding 16-B streams
    // per wave (the 1-row form measured 5.1 TB/s vs the 2-row gateup's 6.4)
    for (int row0 = (blockIdx.x * 4 + wid) * RW; row0 < N;
         row0 += gridDim.x * 4 * RW) {
        const uint32_t* wr[RW];
        bool live[RW];
#pragma unroll
        for (int rr_ = 0; rr_ < RW; ++rr_) {
            live[rr_] = row0 + rr_ < N;
            wr[rr_] = w + (size_t)(live[rr_] ? row0 + rr_ : row0) * k2;
        }
        float acc[RW][M];
#pragma unroll
        for (int rr_ = 0; rr_ < RW; ++rr_)
#pragma unroll
            for (int m = 0; m < M; ++m) acc[rr_][m] = 0.0f;
        for (int i = lane * 4; i < k2; i += WAVE * 4) {
            // stream W non-temporally: each byte is read exactly once per
            // step; keep L2 for the KV cache and activations
            u32x4 wv[RW];
#pragma unroll
            for (int rr_ = 0; rr_ < RW; ++rr_) wv[rr_] = nt_load4(wr[rr_] + i);
#pragma unroll
            for (int m = 0; m < M; ++m) {
                uint4 xv = *reinterpret_cast<const uint4*>(x + (size_t)m * k2 + i);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float xl = bf16_lo((&xv.x)[j]), xh = bf16_hi((&xv.x)[j]);
                    if (NORM) {
                        const uint32_t wnw = wn[i + j];
                        xl *= rstd[m] * bf16_lo(wnw);
                        xh *= rstd[m] * bf16_hi(wnw);
                    }
#pragma unroll
                    for (int rr_ = 0; rr_ < RW; ++rr_) {
                        acc[rr_][m] = fmaf(xl, bf16_lo(wv[rr_][j]), acc[rr_][m]);
                        acc[rr_][m] = fmaf(xh, bf16_hi(wv[rr_][j]), acc[rr_][m]);
                    }
                }
            }
        }
#pragma unroll
        for (int m = 0; m < M; ++m) {
#pragma unroll
            for (int rr_ = 0; rr_ < RW; ++rr_) {
                float v = wave_reduce_sum(acc[rr_][m]);
                if (lane == 0 && live[rr_]) {
                    if (ADDRES) {
                        v += bf16_to_f32(reinterpret_cast<const uint16_t*>(
                            res)[(size_t)m * N + row0 + rr_]);
                    }
                    reinterpret_cast<uint16_t*>(out)[(size_t)m * N + row0 + rr_] =
                        f32_to_bf16(v);
                }
            }
        }
    }
}

// gate activation of the fused gate-up kernels: 0 = silu, 1 = gelu in its tanh
// approximation, g/2 * (1 + tanh(k (g + 0.044715 g^3))), k = sqrt(2/pi)
__device__ __forceinline__ float gate_act(float g, int act) {
    if (act == 1) {
        const float t = tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g));
        return 0.5f * g * (1.0f + t);
    }
    return g / (1.0f + __expf(-g));
}

// Fused gate-up + SiLU GEMV for the MLP up-projection: the fused weight
// holds gate rows [0, I) and up rows [I, 2I); each wave computes BOTH rows
// r and I + r and writes act[m][r] = silu(gate) * up directly — the separate
// [1, 2I] intermediate and the silu_mul pass never materialize.
template <int M, bool NORM>
__global__ __launch_bounds__(256) void gemv_gateup_kernel(
    const uint32_t* __restrict__ x,  // [M, K/2]
    const uint32_t* __restrict__ w,  // [2I, K/2] (gate; up)
    uint32_t* __restrict__ out,      // [M, I] bf16
    const uint32_t* __restrict__ wn, // [K/2] rmsnorm weight (NORM only)
    int I, int k2, float eps, int act) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int wid = threadIdx.x / WAVE;

    float rstd[M];
    if (NORM) {
#pragma unroll
        for (int m = 0; m < M; ++m) rstd[m] = row_rstd(x + (size_t)m * k2, k2, lane, eps);
    }

    for (int row = blockIdx.x * 4 + wid; row < I; row += gridDim.x * 4) {
        const uint32_t* grow = w + (size_t)row * k2;
        const uint32_t* urow = w + (size_t)(I + row) * k2;
        float accg[M], accu[M];
#pragma unroll
        for (int m = 0; m < M; ++m) accg[m] = accu[m] = 0.0f;
        for (int i = lane * 4; i < k2; i += WAVE * 4) {
            u32x4 gv = nt_load4(grow + i);
            u32x4 uv = nt_load4(urow + i);
#pragma unroll
            for (int m = 0; m < M; ++m) {
                uint4 xv = *reinterpret_cast<const uint4*>(x + (size_t)m * k2 + i);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float xl = bf16_lo((&xv.x)[j]), xh = bf16_hi((&xv.x)[j]);
                    if (NORM) {
                        const uint32_t wnw = wn[i + j];
                        xl *= rstd[m] * bf16_lo(wnw);
                        xh *= rstd[m] * bf16_hi(wnw);
                    }
                    accg[m] = fmaf(xl, bf16_lo(gv[j]), accg[m]);
                    accg[m] = fmaf(xh, bf16_hi(gv[j]), accg[m]);
                    accu[m] = fmaf(xl, bf16_lo(uv[j]), accu[m]);
                    accu[m] = fmaf(xh, bf16_hi(uv[j]), accu[m]);
                }
            }
        }
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const float g = wave_reduce_sum(accg[m]);
            const float u = wave_reduce_sum(accu[m]);
            if (lane == 0) {
                const float a = gate_act(g, act) * u;
                reinterpret_cast<uint16_t*>(out)[(size_t)m * I + row] = f32_to_bf16(a);
            }
        }
    }
}

// One activation row (M = 1), K a multiple of 2048. gemv_kernel keeps one 1 KiB load
// per row in flight and, with NORM, normalises the activations again for every row;
// here the block's (normalised) activations are a float32 image in LDS, made while the
// first weight loads are under way, and a wave goes over its rows, every waves-th of the
// weight so that all waves read one window of it (runs of rows instead: 128256 x 2048 93.9
// us, 83.7), as one stream of GR-chunk groups (512 columns each): the next group, also the
// next row's, is loaded before the current one is used. The image keeps columns 0-3 and
// 4-7 of every eight apart, so that 16-byte LDS reads of a wave are contiguous. RT = 2:
// gate and up rows.
// us, gemv_kernel / here, weights of 2 GB in turn: 28672 x 4096 gate-up with norm 43.3 /
// 37.1, 4096 x 14336 25.1 / 20.4, 6144 x 4096 9.6 / 9.9, with norm 12.9 / 10.4, 4096 x 4096
// 8.1 / 7.3, 128256 x 2048 85.3 / 81.2, 2048 x 8192 11.7 / 8.3, 16384 x 2048 gate-up 13.4 /
// 12.7, 2048 x 2048 4.4 / 4.0 (contiguous reads alone run at 6.4 to 6.9 TB/s); asking for
// the activations before the weights takes another half a microsecond each.
//
// EPI 1 adds a residual row. EPI 2 is followed by what dyt_norm (blocks.hip) would do with the bf16
// product y in a launch of its own, 3.2 us for 2048 columns in a chain of launches: r += dyt(y; post),
// out = dyt(r; next) where there is a next norm. A wave's lane i keeps the sum of its row i until all
// are done and then treats that row, for which it asked at the start.
struct DytEpilogue {
    const float *pw, *pb, *pa, *nw, *nb, *na;
    float* residual;
};

// EPI 3 writes the bf16 result as float32 (the logits of a step, us for 32000 x 2048 with the launch that
// would convert them 25.5 / 21.8).
//
// MERGE: the activations are an attention row of heads of D that is still its 2 to 6 key splits (sums o
// [H, splits, D] and maximum and sum of weights ml [H, splits, 2], float32; attn_rows_kernel), which the image
// merges as attn_combine_kernel would: that is a launch of 4.6 us before this one, and every block reads
// all splits, 48 KB of 16 heads of 128, from the L2 while its weights are under way. us, the three launches
// of attention and output product / these two, traced one by one, one row, window 512, 16 heads in 4, 2048 x
// 2048: 16.4 / 13.5; a step of four layers 10 us less. Up to 4096 columns: wider rows have more splits to read than
// the launch takes. Attention and product, us, windows of 512 and contexts of 1400: 16 heads of 128, 2048 x 2048
// 15.1 / 12.9 and 15.7 / 14.6; 32 of 64 13.7 / 11.7 and 15.0 / 12.9; 32 of 128, 4096 x 4096 19.4 / 19.1 and 21.8 / 21.2;
// but 48 of 128, 4096 x 6144 22.6 / 23.9 and 24.5 / 25.7 (6144 x 6144 26.4 / 25.2), 64 of 128, 8192 x 8192 38.0 / 38.4 and
// 39.2 / 40.7.
struct MergeRow {
    const float *o, *ml, *sinks;
    int splits, D;
};

// MORE: MergeRow or nothing, which is no argument (see decode_attn_kernel)
template <bool NORM, int EPI, int RT, int GR, int XV, int WV, typename... MORE>
__global__ __launch_bounds__(WV * 64) void gemv1_kernel(const uint32_t* __restrict__ x,
                                                    const uint32_t* __restrict__ w,
                                                    uint16_t* __restrict__ out,
                                                    const uint32_t* __restrict__ wn,
                                                    const uint16_t* __restrict__ res, int N, int K,
                                                    int waves, int full, int extra, float eps,
                                                    int act, DytEpilogue dy, MORE... more) {
    constexpr bool MERGE = std::is_same_v<void(MORE...), void(MergeRow)>;
    static_assert(MERGE || sizeof...(MORE) == 0, "a row that is merged, or nothing more");
    extern __shared__ __attribute__((aligned(16))) float xl[];   // [2][K / 2]
    __shared__ float part[8];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = blockIdx.x * WV + wid;
    const int k2 = K / 2, groups = K / (512 * GR);
    const int total = (full + (wave < extra)) * groups;     // of the wave's rows: every waves-th
    auto at = [&](int row, int t) { return w + (size_t)(row + (t ? N : 0)) * k2 + lane * 4; };
    u32x4 a[GR][RT], b[GR][RT];
    int row = min(wave, N - 1), g = 0;                      // of the group loaded last
    auto load = [&](u32x4 (&v)[GR][RT]) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int i = 0; i < GR; ++i) v[i][t] = nt_load4(at(row, t) + (g * GR + i) * 256);
    };
    auto next = [&](u32x4 (&v)[GR][RT]) {
        if (++g == groups) {
            g = 0;
            row += waves;
        }
        load(v);
        __builtin_amdgcn_sched_barrier(0);
    };
    // Loads return in order: the activations, eight columns per thread and turn, and lane
    // i's residual of the wave's row i (at most 64) are asked for before the weights, so
    // that the image below waits for them alone.
    uint4 xv[XV], nv[XV];
    constexpr int MS = 6, MX = MERGE ? XV : 1;
    float4 mo[MX][MS][2];
    float2 ms[MX][MS];
    float sink[MX];
#pragma unroll
    for (int j = 0; j < XV; ++j) {
        const int i = min(j * WV * 64 + tid, K / 8 - 1);
        if constexpr (MERGE) {
            const MergeRow mr(more...);
            const int h = i * 8 / mr.D, c = i * 8 - h * mr.D;
#pragma unroll
            for (int s = 0; s < MS; ++s) {
                const int at = h * mr.splits + min(s, mr.splits - 1);
                ms[j][s] = reinterpret_cast<const float2*>(mr.ml)[at];
                const float4* o = reinterpret_cast<const float4*>(mr.o + (size_t)at * mr.D + c);
                mo[j][s][0] = o[0];
                mo[j][s][1] = o[1];
            }
            sink[j] = mr.sinks ? mr.sinks[h] : 0.0f;
            continue;
        }
        xv[j] = reinterpret_cast<const uint4*>(x)[i];
        if (NORM) nv[j] = reinterpret_cast<const uint4*>(wn)[i];
    }
    const int own = (int)min(wave + lane * (int64_t)waves, N - (int64_t)1);
    const float rs = EPI == 1 ? bf16_to_f32(res[own]) : EPI == 2 ? dy.residual[own] : 0.0f;
    float pw = 0, pb = 0, pa = 0, nw = 0, nb = 0, na = 0, mine = 0;
    if constexpr (EPI == 2) {
        pw = dy.pw[own], pb = dy.pb[own], pa = dy.pa[0];
        if (out) nw = dy.nw[own], nb = dy.nb[own], na = dy.na[0];
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
        const int i = j * WV * 64 + tid;
        if (i >= K / 8) continue;
        float f[8];
        if constexpr (MERGE) {
            const MergeRow mr(more...);
            float mx = -INFINITY, l = 0.0f;
#pragma unroll
            for (int s = 0; s < MS; ++s)
                if (s < mr.splits) mx = fmaxf(mx, ms[j][s].x);
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = 0.0f;
#pragma unroll
            for (int s = 0; s < MS; ++s) {
                // (a split without a key has no maximum)
                const float wt = s < mr.splits && ms[j][s].x != -INFINITY ? expf(ms[j][s].x - mx) : 0.0f;
                l += ms[j][s].y * wt;
#pragma unroll
                for (int e = 0; e < 8; ++e) f[e] += (&mo[j][s][e / 4].x)[e % 4] * wt;
            }
            if (mr.sinks) l += expf(sink[j] - mx);
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = bf16_to_f32(f32_to_bf16(f[e] / l));
        }
        if constexpr (!MERGE)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            f[2 * e] = bf16_lo((&xv[j].x)[e]);
            f[2 * e + 1] = bf16_hi((&xv[j].x)[e]);
            if (NORM) {
                f[2 * e] *= rstd * bf16_lo((&nv[j].x)[e]);
                f[2 * e + 1] *= rstd * bf16_hi((&nv[j].x)[e]);
            }
        }
        reinterpret_cast<float4*>(xl)[i] = make_float4(f[0], f[1], f[2], f[3]);
        reinterpret_cast<float4*>(xl + k2)[i] = make_float4(f[4], f[5], f[6], f[7]);
    }
    __syncthreads();

    float acc[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t] = 0.0f;
    int ur = wave, un = 0, ug = 0;                          // of the group in use
    auto use = [&](u32x4 (&v)[GR][RT]) {
#pragma unroll
        for (int i = 0; i < GR; ++i) {
            const int c = (ug * GR + i) * 64 + lane;
            const float4 lo = reinterpret_cast<const float4*>(xl)[c];
            const float4 hi = reinterpret_cast<const float4*>(xl + k2)[c];
#pragma unroll
            for (int t = 0; t < RT; ++t) {
                float s = acc[t];
                s = fmaf(lo.x, bf16_lo(v[i][t][0]), s);
                s = fmaf(lo.y, bf16_hi(v[i][t][0]), s);
                s = fmaf(lo.z, bf16_lo(v[i][t][1]), s);
                s = fmaf(lo.w, bf16_hi(v[i][t][1]), s);
                s = fmaf(hi.x, bf16_lo(v[i][t][2]), s);
                s = fmaf(hi.y, bf16_hi(v[i][t][2]), s);
                s = fmaf(hi.z, bf16_lo(v[i][t][3]), s);
                acc[t] = fmaf(hi.w, bf16_hi(v[i][t][3]), s);
            }
        }
        if (++ug == groups) {
            float v0 = wave_reduce_sum(acc[0]);
            if (RT == 2) v0 = gate_act(v0, act) * wave_reduce_sum(acc[RT - 1]);
            if (EPI == 1)
                v0 += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rs), un));
            if (EPI == 2) mine = lane == un ? v0 : mine;
            else if (EPI == 3 && lane == 0) reinterpret_cast<float*>(out)[ur] = bf16_to_f32(f32_to_bf16(v0));
            else if (lane == 0) out[ur] = f32_to_bf16(v0);
#pragma unroll
            for (int t = 0; t < RT; ++t) acc[t] = 0.0f;
            ug = 0;
            ++un;
            ur += waves;
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
    if constexpr (EPI == 2) {
        if (lane < full + (wave < extra)) {
            const float y = bf16_to_f32(f32_to_bf16(mine)), r = rs + (tanh_f32(pa * y) * pw + pb);
            dy.residual[own] = r;
            if (out) out[own] = f32_to_bf16(tanh_f32(na * r) * nw + nb);
        }
    }
}

// mode as in oa_gemv_ex, 4: dy; 5: out float32; gateup > 0: N gate and N up rows, activation gateup - 1
static int gemv1(hipStream_t st, const void* x, const void* w, void* out, const void* wn,
                 const void* res, int N, int K, float eps, int mode, int gateup,
                 const DytEpilogue& dy = {}, const MergeRow& mr = {}) {
    // Rows of 4096, and many of 2048: blocks of four waves, of two rows a wave (gate-up one
    // pair), so that CUs even out; the image of a block is quickly made. No more than 32
    // blocks per CU. Us, blocks of eight waves and up to 64 rows a wave / this: 6144 x 4096
    // 10.4 / 9.9, 4096 x 4096 8.5 / 7.3, 32000 x 4096 43.5 / 40.8, 2 x 14336 x 4096 38.4 /
    // 36.4, 128256 x 2048 83.4 / 78.2, 2 x 2816 x 2048 6.6 / 6.3, but 2048 x 2048 3.9 / 4.2, 2
    // x 1408 x 2048 4.5 / 5.0, 2 x 8192 x 2048 12.7 / 12.9.
    // Else: as many blocks of eight waves as stay resident (two per CU by registers, four
    // with short rows), fewer and fuller ones where that evens out the CUs by more than a
    // fifth.
    // A norm makes the image of every block dearer: with one, gate-up of up to 8192 rows and
    // few plain rows stay with eight waves (us, eight / four: 2 x 4096 x 4096 12.5 / 13.8, 2
    // x 1408 x 4096 5.8 / 7.0, 2 x 9216 x 4096 27.4 / 26.2; 512 x 4096 4.2 / 4.5, 2048 x 4096
    // 5.1 / 4.8).
    const bool dear = (mode & 1) && (gateup ? N <= 8192 : N <= 1024);
    const int wv = (K == 4096 && !dear) || (K == 2048 && (gateup ? N > 2048 && N <= 4096 : N > 4096)) ? 4 : 8;
    int per;
    if (wv == 4) {
        per = CEIL_DIV(N, 256 * 4 * 32);
        // one row a wave where two leave CUs uneven by a sixth (us, two / one: 5120 x 4096 9.8 /
        // 9.5, 3072 x 4096 7.0 / 6.6, 512 x 4096 4.6 / 3.8)
        const int one = CEIL_DIV(CEIL_DIV(N, 4), 256), two = 2 * CEIL_DIV(CEIL_DIV(N, 8), 256);
        if (!gateup && per < 2 && two * 5 < one * 6) per = 2;
    } else {
        auto rounds = [&](int p) { return CEIL_DIV(CEIL_DIV(CEIL_DIV(N, p), 8), 256) * p; };
        per = CEIL_DIV(N, 2048 * (K == 2048 && !gateup ? 4 : 2));
        for (int p = per + 1, p1 = 2 * per + 1; p <= p1; ++p)
            if (rounds(p) * 5 < rounds(per) * 4) per = p;
    }
    if (per > 64) per = 64;
    const int blocks = CEIL_DIV(CEIL_DIV(N, per), wv);
    const int waves = blocks * wv;
    const size_t lds = (size_t)K * 4;
#define G1X(NV, RV, RT, GR, XV, WV, ...)                                                              \
    hipLaunchKernelGGL((gemv1_kernel<NV, RV, RT, GR, XV, WV>), dim3(blocks), dim3(WV * 64), lds, st,  \
                       (const uint32_t*)x, (const uint32_t*)w, (uint16_t*)out, (const uint32_t*)wn,   \
                       (const uint16_t*)res, N, K, waves, N / waves, N % waves, eps, gateup - 1, dy,  \
                       ##__VA_ARGS__)
#define G1(NV, RV, RT, GR)                   \
    do {                                     \
        if (wv == 4) G1X(NV, RV, RT, GR, 2, 4);         \
        else if (K <= 4096) G1X(NV, RV, RT, GR, 1, 8);  \
        else G1X(NV, RV, RT, GR, 4, 8);                 \
    } while (0)
    if (mr.o) {                          // K up to 4096
        if (K == 4096) G1X(false, 2, 1, 8, 2, 4, mr);
        else if (wv == 4) G1X(false, 2, 1, 4, 2, 4, mr);
        else G1X(false, 2, 1, 4, 1, 8, mr);
    } else if (gateup) {
        if (mode & 1) G1(true, 0, 2, 4);
        else G1(false, 0, 2, 4);
    } else if (K % 4096 == 0) {
        switch (mode) {
            case 0: G1(false, 0, 1, 8); break;
            case 1: G1(true, 0, 1, 8); break;
            case 2: G1(false, 1, 1, 8); break;
            case 3: G1(true, 1, 1, 8); break;
            case 5: G1(false, 3, 1, 8); break;
            default: G1(false, 2, 1, 8); break;
        }
    } else {
        switch (mode) {
            case 0: G1(false, 0, 1, 4); break;
            case 1: G1(true, 0, 1, 4); break;
            case 2: G1(false, 1, 1, 4); break;
            case 3: G1(true, 1, 1, 4); break;
            case 5: G1(false, 3, 1, 4); break;
            default: G1(false, 2, 1, 4); break;
        }
    }
#undef G1
#undef G1X
    HIP_CHECK_LAUNCH();
    return 0;
}
// the float32 image of the activations fits the LDS of two blocks per CU
static bool gemv1_ok(int M, int K) { return M == 1 && K % 2048 == 0 && K <= 16384; }

// residual += dyt(x W^T; pw, pb, pa), out = dyt(residual; nw, nb, na) unless null: one row x [K],
// residual [N] and the norms float32 (pa, na: one number each); nothing where gemv1 does not take it
extern "C" int oa_gemv_dyt(void* stream, const void* x, const void* w, void* residual, const void* pw,
                           const void* pb, const void* pa, const void* nw, const void* nb, const void* na,
                           void* out, int N, int K) {
    if (N < 1 || !gemv1_ok(1, K) || N > 256 * 64 * 8) return -100;
    if (!x || !w || !residual || !pw || !pb || !pa || (out && (!nw || !nb || !na))) return -101;
    if (((uintptr_t)x | (uintptr_t)w) % 16 != 0) return -102;
    const DytEpilogue dy = {(const float*)pw, (const float*)pb, (const float*)pa, (const float*)nw,
                            (const float*)nb, (const float*)na, (float*)residual};
    return gemv1((hipStream_t)stream, x, w, out, nullptr, nullptr, N, K, 0.0f, 4, 0, dy);
}

static bool gemv_bf16_use_mfma(int M, int K, int gateup);
extern "C" int oa_gemv_bf16_mfma(void* stream, const void* x, const void* w,
                                 void* out, const void* wn, const void* res,
                                 int M, int N, int K, float eps, int mode,
                                 int gateup);

static int gemv_gateup_impl(void* stream, const void* x, const void* w,
                            void* out, const void* wn, int M, int I, int K,
                            float eps, int norm, int act) {
    if (K % 8 != 0) return -100;
    if (gemv1_ok(M, K))
        return gemv1((hipStream_t)stream, x, w, out, wn, nullptr, I, K, eps, norm ? 1 : 0, 1 + act);
    if (gemv_bf16_use_mfma(M, K, 1))
        return oa_gemv_bf16_mfma(stream, x, w, out, wn, nullptr, M, 2 * I, K,
                                 eps, norm ? 1 : 0, 1 + act);
    const int k2 = K / 2;
    const int grid = min(2048, CEIL_DIV(I, 4));
#define LAUNCH_GU(MV)                                                          \
    do {                                                                       \
        if (norm)                                                              \
            hipLaunchKernelGGL((gemv_gateup_kernel<MV, true>), dim3(grid),     \
                               dim3(256), 0, (hipStream_t)stream,              \
                               (const uint32_t*)x, (const uint32_t*)w,         \
                               (uint32_t*)out, (const uint32_t*)wn, I, k2, eps, act);\
        else                                                                   \
            hipLaunchKernelGGL((gemv_gateup_kernel<MV, false>), dim3(grid),    \
                               dim3(256), 0, (hipStream_t)stream,              \
                               (const uint32_t*)x, (const uint32_t*)w,         \
                               (uint32_t*)out, (const uint32_t*)wn, I, k2, eps, act);\
    } while (0)
    switch (M) {
        case 1: LAUNCH_GU(1); break;
        case 2: LAUNCH_GU(2); break;
        case 3: LAUNCH_GU(3); break;
        case 4: LAUNCH_GU(4); break;
        case 5: LAUNCH_GU(5); break;
        case 6: LAUNCH_GU(6); break;
        case 7: LAUNCH_GU(7); break;
        case 8: LAUNCH_GU(8); break;
        case 12: LAUNCH_GU(12); break;
        case 16: LAUNCH_GU(16); break;
        default: return -101;
    }
#undef LAUNCH_GU
    HIP_CHECK_LAUNCH();
    return 0;
}

extern "C" int oa_gemv_gateup_ex(void* stream, const void* x, const void* w,
                                 void* out, const void* wn, int M, int I, int K,
                                 float eps, int norm) {
    return gemv_gateup_impl(stream, x, w, out, wn, M, I, K, eps, norm, 0);
}

// act: 0 silu, 1 gelu (tanh form)
extern "C" int oa_gemv_gateup_act(void* stream, const void* x, const void* w,
                                  void* out, int M, int I, int K, int act) {
    if (act < 0 || act > 1) return -105;
    return gemv_gateup_impl(stream, x, w, out, nullptr, M, I, K, 0.0f, 0, act);
}

// mode: 0 plain, 1 norm-prologue, 2 residual-add epilogue, 3 both
// out [N] float32 = bf16(x W^T), one row
extern "C" int oa_gemv_float(void* stream, const void* x, const void* w, void* out, int N, int K) {
    if (N < 1 || !gemv1_ok(1, K)) return -100;
    if (!x || !w || !out) return -101;
    if (((uintptr_t)x | (uintptr_t)w) % 16 != 0) return -102;
    return gemv1((hipStream_t)stream, x, w, out, nullptr, nullptr, N, K, 0.0f, 5, 0);
}

// oa_gemv_dyt of a row that is still its key splits (MergeRow): K up to 4096, heads of 64 or 128
extern "C" int oa_gemv_dyt_merge(void* stream, const void* o, const void* ml, const void* sinks, int splits, int D,
                                 const void* w, void* residual, const void* pw, const void* pb, const void* pa,
                                 const void* nw, const void* nb, const void* na, void* out, int N, int K) {
    if (N < 1 || K < 2048 || K % 2048 != 0 || K > 4096 || N > 256 * 64 * 8) return -100;
    if (splits < 2 || splits > 6 || (D != 64 && D != 128)) return -103;
    if (!o || !ml || !w || !residual || !pw || !pb || !pa || (out && (!nw || !nb || !na))) return -101;
    if (((uintptr_t)o | (uintptr_t)w) % 16 != 0 || (uintptr_t)ml % 8 != 0) return -102;
    const DytEpilogue dy = {(const float*)pw, (const float*)pb, (const float*)pa, (const float*)nw,
                            (const float*)nb, (const float*)na, (float*)residual};
    const MergeRow mr = {(const float*)o, (const float*)ml, (const float*)sinks, splits, D};
    return gemv1((hipStream_t)stream, nullptr, w, out, nullptr, nullptr, N, K, 0.0f, 4, 0, dy, mr);
}

extern "C" int oa_gemv_ex(void* stream, const void* x, const void* w, void* out,
                          const void* wn, const void* res, int M, int N, int K,
                          float eps, int mode) {
    if (K % 8 != 0) return -100;
    if (mode < 0 || mode > 3) return -102;
    if (gemv1_ok(M, K)) return gemv1((hipStream_t)stream, x, w, out, wn, res, N, K, eps, mode, 0);
    if (gemv_bf16_use_mfma(M, K, 0))
        return oa_gemv_bf16_mfma(stream, x, w, out, wn, res, M, N, K, eps,
                                 mode, 0);
    const int k2 = K / 2;
    // 4 rows/wave won +3-6% in the ISOLATED probe on wide outputs
    // (scripts/gemv_ab.py) but lost 3% in-model (decode step 3.63 -> 3.75 ms,
    // within-box A/B) — real decode interleaves the W stream with KV/L2
    // traffic the probe does not. Default OFF; OPSAGENT_GEMV_RW4_MIN_N
    // re-enables for experiments.
    static int rw4_min_n = -1;
    static int rw1_max_n = -1;
    if (rw4_min_n < 0) {
        const char* e = getenv("OPSAGENT_GEMV_RW4_MIN_N");
        rw4_min_n = e ? atoi(e) : (1 << 30);
        // RW=1 for small-N outputs: at N=4096 the RW=2 grid is only 512
        // workgroups (2 per CU — half the SIMD slots idle); one row per wave
        // doubles the wave count and the streams in flight. In-model A/B
        // (8B turn, same box): off 438.1 ms, N<=6144 431.0 ms, N<=4096
        // 431.9 ms — default N<=6144 (covers o_proj and the fused-norm qkv).
        const char* e1 = getenv("OPSAGENT_GEMV_RW1_MAX_N");
        rw1_max_n = e1 ? atoi(e1) : 6144;
    }
    const bool rw4 = N >= rw4_min_n;
    const bool rw1 = !rw4 && N <= rw1_max_n;
    const int grid = min(2048, CEIL_DIV(N, rw4 ? 16 : (rw1 ? 4 : 8)));
#define LAUNCH_NM(MV, NORMV, RESV)                                            \
    do {                                                                       \
        if (rw4)                                                               \
            hipLaunchKernelGGL((gemv_kernel<MV, NORMV, RESV, 4>), dim3(grid),  \
                               dim3(256), 0, (hipStream_t)stream,              \
                               (const uint32_t*)x, (const uint32_t*)w,         \
                               (uint32_t*)out, (const uint32_t*)wn,            \
                               (const uint32_t*)res, N, k2, eps);              \
        else if (rw1)                                                          \
            hipLaunchKernelGGL((gemv_kernel<MV, NORMV, RESV, 1>), dim3(grid),  \
                               dim3(256), 0, (hipStream_t)stream,              \
                               (const uint32_t*)x, (const uint32_t*)w,         \
                               (uint32_t*)out, (const uint32_t*)wn,            \
                               (const uint32_t*)res, N, k2, eps);              \
        else                                                                   \
            hipLaunchKernelGGL((gemv_kernel<MV, NORMV, RESV, 2>), dim3(grid),  \
                               dim3(256), 0, (hipStream_t)stream,              \
                               (const uint32_t*)x, (const uint32_t*)w,         \
                               (uint32_t*)out, (const uint32_t*)wn,            \
                               (const uint32_t*)res, N, k2, eps);              \
    } while (0)
#define LAUNCH_MODE(MV)                                                        \
    do {                                                                       \
        switch (mode) {                                                        \
            case 0: LAUNCH_NM(MV, false, false); break;                        \
            case 1: LAUNCH_NM(MV, true, false); break;                         \
            case 2: LAUNCH_NM(MV, false, true); break;                         \
            case 3: LAUNCH_NM(MV, true, true); break;                          \
            default: return -102;                                              \
        }                                                                      \
    } while (0)
    switch (M) {
        case 1: LAUNCH_MODE(1); break;
        case 2: LAUNCH_MODE(2); break;
        case 3: LAUNCH_MODE(3); break;
        case 4: LAUNCH_MODE(4); break;
        case 5: LAUNCH_MODE(5); break;
        case 6: LAUNCH_MODE(6); break;
        case 7: LAUNCH_MODE(7); break;
        case 8: LAUNCH_MODE(8); break;
        case 12: LAUNCH_MODE(12); break;
        case 16: LAUNCH_MODE(16); break;
        default: return -101;
    }
#undef LAUNCH_MODE
#undef LAUNCH_NM
    HIP_CHECK_LAUNCH();
    return 0;
}

extern "C" int oa_gemv(void* stream, const void* x, const void* w, void* out,
                       int M, int N, int K) {
    return oa_gemv_ex(stream, x, w, out, nullptr, nullptr, M, N, K, 0.0f, 0);
}

// RW=4 probe variant (within-probe A/B only)
extern "C" int oa_gemv_rw4(void* stream, const void* x, const void* w, void* out,
                           int M, int N, int K) {
    if (K % 8 != 0) return -100;
    const int k2 = K / 2;
    const int grid = min(2048, CEIL_DIV(N, 16));
    switch (M) {
        case 1:
            hipLaunchKernelGGL((gemv_kernel<1, false, false, 4>), dim3(grid),
                               dim3(256), 0, (hipStream_t)stream,
                               (const uint32_t*)x, (const uint32_t*)w,
                               (uint32_t*)out, nullptr, nullptr, N, k2, 0.0f);
            break;
        default:
            return -101;
    }
    HIP_CHECK_LAUNCH();
    return 0;
}

// ---- MFMA bf16 GEMV (batched decode, M 2..16) ------------------------------
// The VALU kernels win at M <= 2 but their per-element M-loop turns
// compute-bound as the batch grows, and hipBLASLt's skinny kernels (the old
// M > 2 fallback) run ~2.5x off the stream roofline — concurrent decode
// (c=8/16) measured ~2 TB/s effective. Same architecture as the fp8 MFMA
// GEMV (fp8_moe.hip): x staged ONCE into LDS (norm applied in fp32 at stage
// time), each of the block's four waves streams 16 W rows over a quarter of
// K straight into v_mfma_f32_16x16x32_bf16 A-fragments with a PF-deep
// register prefetch ring, partial D tiles meet in LDS. The 16 B columns
// carry the batch — M up to 16 rides one weight stream.
typedef __attribute__((ext_vector_type(8))) short bf16x8g;
typedef __attribute__((ext_vector_type(4))) float f32x4g;

template <bool NORM, bool ADDRES, bool GATEUP>
__global__ __launch_bounds__(256, 1) void gemv_bf16_mfma_kernel(
    const uint32_t* __restrict__ x,   // [M, K/2] bf16x2
    const uint32_t* __restrict__ w,   // [N, K/2] (gateup: [2I, K/2])
    uint32_t* __restrict__ out,       // [M, N] bf16 (gateup: [M, I])
    const uint32_t* __restrict__ wn,  // [K/2] rmsnorm weight (NORM)
    const uint32_t* __restrict__ res, // [M, N] residual (ADDRES)
    int M, int N, int K, float eps, int act) {
    constexpr int PF = GATEUP ? 4 : 8;
    const int tid = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int wid = tid / WAVE;
    const int fr = lane & 15;   // A row / B,D col
    const int fs = lane >> 4;   // 8-element k-slice; D rows fs*4..+3
    const int rows = GATEUP ? N / 2 : N;
    const int I = rows;
    const int row0 = blockIdx.x * 16;
    const int wrow = min(row0 + fr, rows - 1);
    const int k2 = K / 2;

    extern __shared__ __attribute__((aligned(16))) char xls[];
    const int pitch = K * 2 + 16;  // bytes; pad de-banks the batch rows

    // stage x (wave w handles batch rows m ≡ w mod 4), norm folded in fp32
    for (int m = wid; m < M; m += 4) {
        const uint32_t* xr = x + (size_t)m * k2;
        uint32_t* dst = reinterpret_cast<uint32_t*>(xls + (size_t)m * pitch);
        float rstd = 1.0f;
        if (NORM) rstd = row_rstd(xr, k2, lane, eps);
        for (int i = lane * 4; i < k2; i += WAVE * 4) {
            uint4 v = *reinterpret_cast<const uint4*>(xr + i);
            if (NORM) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t g = wn[i + j];
                    const float lo = bf16_lo((&v.x)[j]) * rstd * bf16_lo(g);
                    const float hi = bf16_hi((&v.x)[j]) * rstd * bf16_hi(g);
                    (&v.x)[j] = (uint32_t)f32_to_bf16(lo) |
                                ((uint32_t)f32_to_bf16(hi) << 16);
                }
            }
            *reinterpret_cast<uint4*>(dst + i) = v;
        }
    }
    __syncthreads();

    const int ke = K / 4;               // elements per wave
    const int k0b = wid * ke * 2;       // byte offset of this wave's range
    const int nk = ke / 32;             // 32-element MFMA steps
    const char* wp = reinterpret_cast<const char*>(w);
    const uint32_t* wr0 = reinterpret_cast<const uint32_t*>(
        wp + (size_t)wrow * K * 2 + k0b) + fs * 4;
    const uint32_t* wr1 = reinterpret_cast<const uint32_t*>(
        wp + (size_t)(wrow + (GATEUP ? I : 0)) * K * 2 + k0b) + fs * 4;
    const int mrow = fr < M ? fr : 0;
    const char* xrw = xls + (size_t)mrow * pitch + k0b + fs * 16;

    f32x4g acc0 = {}, acc1 = {};
    uint4 abuf[PF], ubuf[GATEUP ? PF : 1];
    auto load_a = [&](int p, int kb) {
        u32x4 t = nt_load4(wr0 + kb * 16);
        abuf[p] = *reinterpret_cast<uint4*>(&t);
        if (GATEUP) {
            u32x4 t2 = nt_load4(wr1 + kb * 16);
            ubuf[p] = *reinterpret_cast<uint4*>(&t2);
        }
    };
#pragma unroll
    for (int p = 0; p < PF; ++p) load_a(p, p);
    // x fragment double-buffered ONE step ahead: an inline ds_read feeding
    // its own MFMA serializes on lgkmcnt(0) every step (measured in the .s)
    uint4 bcur = *reinterpret_cast<const uint4*>(xrw);
    for (int kb0 = 0; kb0 < nk; kb0 += PF) {
        const bool more = kb0 + PF < nk;
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            const int kb = kb0 + p;
            uint4 bnext;
            if (kb + 1 < nk)
                bnext = *reinterpret_cast<const uint4*>(xrw + (kb + 1) * 64);
            acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                *reinterpret_cast<bf16x8g*>(&abuf[p]),
                *reinterpret_cast<bf16x8g*>(&bcur), acc0, 0, 0, 0);
            if (GATEUP)
                acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    *reinterpret_cast<bf16x8g*>(&ubuf[p]),
                    *reinterpret_cast<bf16x8g*>(&bcur), acc1, 0, 0, 0);
            if (more) load_a(p, kb0 + PF + p);
            if (kb + 1 < nk) bcur = bnext;
        }
    }

    // intra-block reduction: [wave][plane][col fr][row fs*4+i] f32 in LDS
    __syncthreads();  // x reads done before the tiles overwrite the image
    float* red = reinterpret_cast<float*>(xls);
    const int planes = GATEUP ? 2 : 1;
    {
        float* t = red + ((wid * planes) * 16 + fr) * 16 + fs * 4;
        *reinterpret_cast<f32x4g*>(t) = acc0;
        if (GATEUP) *reinterpret_cast<f32x4g*>(t + 16 * 16) = acc1;
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
        for (int wv = 0; wv < 4; ++wv) {
            sg += red[((wv * planes) * 16 + m) * 16 + fs * 4 + i];
            if (GATEUP)
                su += red[((wv * planes + 1) * 16 + m) * 16 + fs * 4 + i];
        }
        float v;
        if (GATEUP) {
            v = gate_act(sg, act) * su;
        } else {
            v = sg;
            if (ADDRES)
                v += bf16_to_f32(reinterpret_cast<const uint16_t*>(
                    res)[(size_t)m * rows + row]);
        }
        reinterpret_cast<uint16_t*>(out)[(size_t)m * rows + row] =
            f32_to_bf16(v);
    }
}

// eligibility shared by the C dispatch and its callers; must mirror the
// kernel's constraints so ineligible shapes FALL BACK, never error
static bool gemv_bf16_use_mfma(int M, int K, int gateup) {
    const char* e = getenv("OPSAGENT_BF16_GEMV_MFMA");
    if (e && e[0] == '0') return false;
    int min_m = 3;  // VALU kernels keep the measured M<=2 regime
    if (e && e[0] == 'm') min_m = atoi(e + 1);
    if (M < min_m || M > 16) return false;
    if (K % (gateup ? 512 : 1024) != 0) return false;
    // A/B-measured win region (scripts/gemv_bf16_mfma_ab.py): +29..+83%
    // at the 8B-class K<=6144 shapes; hipBLASLt keeps deep-K (70B qkv
    // K=8192 5.56 TB/s vs 3.21; 8B down K=14336 a wash) and the M=16
    // gateup (131 KiB x-image halves block occupancy). Env 'm<N>' widens
    // for experiments.
    if (!(e && e[0] == 'm')) {
        // engine A/B at c16 (same box): the M 9..16 forms LOSE ~7% end to
        // end even though the M16 microbench won — cap at the regime both
        // agree on (M <= 8, K <= 6144)
        if (K > 6144 || M > 8) return false;
    }
    const size_t img = (size_t)M * (K * 2 + 16);
    return img <= 147456;
}

extern "C" int oa_gemv_bf16_mfma(void* stream, const void* x, const void* w,
                                 void* out, const void* wn, const void* res,
                                 int M, int N, int K, float eps, int mode,
                                 int gateup) {
    const int rows = gateup ? N / 2 : N;
    const size_t img = (size_t)M * (K * 2 + 16);
    const size_t red = (size_t)(gateup ? 2 : 1) * 4 * 16 * 16 * 4;
    const size_t shmem = img > red ? img : red;
    dim3 grid(CEIL_DIV(rows, 16)), block(256);
#define LAUNCH_BMF(NORMV, RESV, GUV)                                           \
    hipLaunchKernelGGL((gemv_bf16_mfma_kernel<NORMV, RESV, GUV>), grid, block, \
                       shmem, (hipStream_t)stream, (const uint32_t*)x,         \
                       (const uint32_t*)w, (uint32_t*)out,                     \
                       (const uint32_t*)wn, (const uint32_t*)res, M, N, K, eps, \
                       gateup > 1 ? gateup - 1 : 0)
    if (gateup) {
        if (mode & 1) LAUNCH_BMF(true, false, true);
        else LAUNCH_BMF(false, false, true);
    } else {
        switch (mode) {
            case 0: LAUNCH_BMF(false, false, false); break;
            case 1: LAUNCH_BMF(true, false, false); break;
            case 2: LAUNCH_BMF(false, true, false); break;
            case 3: LAUNCH_BMF(true, true, false); break;
            default: return -102;
        }
    }
#undef LAUNCH_BMF
    HIP_CHECK_LAUNCH();
    return 0;
}

// ---- grouped rows -----------------------------------------------------------
// One launch for all projections of a layer that read the same normed input or
// per-projection variants of it: the weight's rows [N, K] are cut into groups,
// group g = rows [begin, end), reads activation plane `plane` of x [P, M, K]
// and writes act(row . x) to column row - begin of its own output rows.
// begin and end are multiples of 16, so neither the two adjacent rows of a
// wave nor the 16 rows of a matrix-core tile straddle a group. In a paired group
// gate and up rows alternate and (row - begin) / 2 takes act(gate) * up.
#define GEMV_MAX_GROUPS 8
struct GemvGroups {
    int n;
    int end[GEMV_MAX_GROUPS];
    int plane[GEMV_MAX_GROUPS];
    int act[GEMV_MAX_GROUPS];         // 0 none, 1 silu, 2 gelu (tanh form); + 4: paired
    uint16_t* out[GEMV_MAX_GROUPS];
    int64_t os[GEMV_MAX_GROUPS];      // elements between the output rows
};

__device__ __forceinline__ int gemv_group_of(const GemvGroups& g, int row) {
    int k = 0;
    while (k + 1 < g.n && row >= g.end[k]) ++k;
    return k;
}
__device__ __forceinline__ float gemv_group_act(float v, int act) {
    return act ? gate_act(v, act - 1) : v;
}
#define GEMV_PAIRED 4

template <int M, int RW>
__global__ __launch_bounds__(256) void gemv_grouped_kernel(const uint32_t* __restrict__ x,
                                                           const uint32_t* __restrict__ w,
                                                           GemvGroups gr, int N, int k2) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    for (int row0 = (blockIdx.x * 4 + wid) * RW; row0 < N; row0 += gridDim.x * 4 * RW) {
        const int gi = gemv_group_of(gr, row0);
        const uint32_t* xg = x + (size_t)gr.plane[gi] * M * k2;
        const uint32_t* wr = w + (size_t)row0 * k2;
        float acc[RW][M];
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
            for (int m = 0; m < M; ++m) acc[r][m] = 0.0f;
        for (int i = lane * 4; i < k2; i += WAVE * 4) {
            u32x4 wv[RW];
#pragma unroll
            for (int r = 0; r < RW; ++r) wv[r] = nt_load4(wr + (size_t)r * k2 + i);
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const uint4 xv = *reinterpret_cast<const uint4*>(xg + (size_t)m * k2 + i);
                const uint32_t xs[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float xl = bf16_lo(xs[j]), xh = bf16_hi(xs[j]);
#pragma unroll
                    for (int r = 0; r < RW; ++r) {
                        acc[r][m] = fmaf(xl, bf16_lo(wv[r][j]), acc[r][m]);
                        acc[r][m] = fmaf(xh, bf16_hi(wv[r][j]), acc[r][m]);
                    }
                }
            }
        }
        const int c0 = row0 - (gi ? gr.end[gi - 1] : 0);
        uint16_t* out = gr.out[gi];
        if (RW == 2 && (gr.act[gi] & GEMV_PAIRED)) {
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const float g = wave_reduce_sum(acc[0][m]), u = wave_reduce_sum(acc[RW - 1][m]);
                if (lane == 0)
                    out[(size_t)m * gr.os[gi] + c0 / 2] =
                        f32_to_bf16(gemv_group_act(g, gr.act[gi] - GEMV_PAIRED) * u);
            }
            continue;
        }
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                const float v = wave_reduce_sum(acc[r][m]);
                if (lane == 0)
                    out[(size_t)m * gr.os[gi] + c0 + r] = f32_to_bf16(gemv_group_act(v, gr.act[gi]));
            }
    }
}

// The matrix-core form: see gemv_bf16_mfma_kernel for the tiling. SPLIT: one
// group, K cut into pieces of `unit` columns over gridDim.y blocks; a block
// writes its float32 partial sums to part [gridDim.y, M, N], and the kernel
// that reads the product adds the pieces up. A deep K thereby fits the LDS
// image of the activations and fills the chip.
template <bool SPLIT>
__global__ __launch_bounds__(256, 1) void gemv_grouped_mfma_kernel(
    const uint32_t* __restrict__ x, const uint32_t* __restrict__ w, GemvGroups gr, int M, int K,
    int unit, float* __restrict__ part) {
    constexpr int PF = 8;
    const int tid = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int wid = tid / WAVE;
    const int fr = lane & 15, fs = lane >> 4;
    const int row0 = blockIdx.x * 16;
    const int gi = SPLIT ? 0 : gemv_group_of(gr, row0);
    const int k2 = K / 2;
    const int kb_ = SPLIT ? blockIdx.y * unit : 0;       // first column of this block
    const int kl = SPLIT ? min(unit, K - kb_) : K;       // its columns, a multiple of 1024
    extern __shared__ __attribute__((aligned(16))) char xls[];
    const int pitch = kl * 2 + 16;
    const uint32_t* xg = x + (size_t)(SPLIT ? 0 : gr.plane[gi]) * M * k2 + kb_ / 2;
    const int ke = kl / 4;
    const int k0b = wid * ke * 2;
    const int nk = ke / 32;             // a multiple of PF
    const uint32_t* wr = reinterpret_cast<const uint32_t*>(
        reinterpret_cast<const char*>(w) + ((size_t)(row0 + fr) * K + kb_) * 2 + k0b) + fs * 4;
    u32x4 abuf[PF];
#pragma unroll
    for (int p = 0; p < PF; ++p) abuf[p] = nt_load4(wr + p * 16);
    for (int m = wid; m < M; m += 4) {
        const uint32_t* xr = xg + (size_t)m * k2;
        uint32_t* dst = reinterpret_cast<uint32_t*>(xls + (size_t)m * pitch);
        for (int i = lane * 4; i < kl / 2; i += WAVE * 4)
            *reinterpret_cast<uint4*>(dst + i) = *reinterpret_cast<const uint4*>(xr + i);
    }
    __syncthreads();
    const char* xrw = xls + (size_t)(fr < M ? fr : 0) * pitch + k0b + fs * 16;
    f32x4g acc = {};
    uint4 bcur = *reinterpret_cast<const uint4*>(xrw);
    for (int kb0 = 0; kb0 < nk; kb0 += PF) {
        const bool more = kb0 + PF < nk;
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            const int kb = kb0 + p;
            uint4 bnext = bcur;
            if (kb + 1 < nk) bnext = *reinterpret_cast<const uint4*>(xrw + (kb + 1) * 64);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<bf16x8g*>(&abuf[p]),
                                                          *reinterpret_cast<bf16x8g*>(&bcur), acc, 0, 0, 0);
            if (more) abuf[p] = nt_load4(wr + (kb0 + PF + p) * 16);
            bcur = bnext;
        }
    }
    __syncthreads();   // x reads done before the partial tiles overwrite the image
    float* red = reinterpret_cast<float*>(xls);
    *reinterpret_cast<f32x4g*>(red + (wid * 16 + fr) * 16 + fs * 4) = acc;
    __syncthreads();
    if (wid != 0 || fr >= M) return;
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[i] = 0.0f;
#pragma unroll
        for (int wv = 0; wv < 4; ++wv) v[i] += red[(wv * 16 + fr) * 16 + fs * 4 + i];
    }
    if (SPLIT) {
        const int N = gridDim.x * 16;
        *reinterpret_cast<float4*>(part + ((size_t)blockIdx.y * M + fr) * N + row0 + fs * 4) =
            make_float4(v[0], v[1], v[2], v[3]);
        return;
    }
    const int c0 = row0 - (gi ? gr.end[gi - 1] : 0);
    if (gr.act[gi] & GEMV_PAIRED) {
        uint16_t* po = gr.out[gi] + (size_t)fr * gr.os[gi] + c0 / 2 + fs * 2;
        const int act = gr.act[gi] - GEMV_PAIRED;
#pragma unroll
        for (int i = 0; i < 2; ++i) po[i] = f32_to_bf16(gemv_group_act(v[2 * i], act) * v[2 * i + 1]);
        return;
    }
    uint16_t* out = gr.out[gi] + (size_t)fr * gr.os[gi] + c0 + fs * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = f32_to_bf16(gemv_group_act(v[i], gr.act[gi]));
}

// Partial sums of x [M, K] @ w [N, K]^T: part [ceil(K / unit), M, N] float32.
// K and unit multiples of 1024, N of 16, M <= 16.
extern "C" int oa_gemv_split(void* stream, const void* x, const void* w, void* part, int M, int N, int K,
                             int unit) {
    if (M < 1 || M > 16 || N % 16 != 0 || K % 1024 != 0 || unit < 1024 || unit % 1024 != 0) return -100;
    const size_t img = (size_t)M * (std::min(unit, K) * 2 + 16), red = 4 * 16 * 16 * 4;
    if (img > 147456) return -104;
    GemvGroups none = {};
    hipLaunchKernelGGL(gemv_grouped_mfma_kernel<true>, dim3(N / 16, CEIL_DIV(K, unit)), dim3(256),
                       img > red ? img : red, (hipStream_t)stream, (const uint32_t*)x,
                       (const uint32_t*)w, none, M, K, unit, (float*)part);
    HIP_CHECK_LAUNCH();
    return 0;
}

// x [P, M, K] contiguous (every group's plane < P, checked by the caller);
// w [N, K]; end/plane/act/out/os: host arrays of n entries, end[n-1] = N.
// mfma: the matrix-core form (K % 1024 == 0, M <= 16), else M 1..4.
extern "C" int oa_gemv_grouped(void* stream, const void* x, const void* w, int M, int N, int K, int n,
                               const int* end, const int* plane, const int* act, void* const* out,
                               const int64_t* os, int mfma) {
    if (M < 1 || n < 1 || n > GEMV_MAX_GROUPS || K % 8 != 0) return -100;
    GemvGroups gr;
    gr.n = n;
    int prev = 0;
    bool paired = false;
    for (int i = 0; i < n; ++i) {
        const int kind = act[i] & ~GEMV_PAIRED, pair = act[i] & GEMV_PAIRED ? 1 : 0;
        if (end[i] <= prev || end[i] % 16 != 0 || plane[i] < 0 || kind < 0 || kind > 2 || !out[i] ||
            os[i] < (end[i] - prev) >> pair)
            return -101;
        paired |= pair;
        gr.end[i] = prev = end[i];
        gr.plane[i] = plane[i];
        gr.act[i] = act[i];
        gr.out[i] = (uint16_t*)out[i];
        gr.os[i] = os[i];
    }
    if (prev != N) return -102;
    hipStream_t s = (hipStream_t)stream;
    if (mfma) {
        if (M > 16 || K % 1024 != 0) return -103;
        const size_t img = (size_t)M * (K * 2 + 16), red = 4 * 16 * 16 * 4;
        if (img > 147456) return -104;
        hipLaunchKernelGGL(gemv_grouped_mfma_kernel<false>, dim3(N / 16), dim3(256), img > red ? img : red,
                           s, (const uint32_t*)x, (const uint32_t*)w, gr, M, K, K, (float*)nullptr);
        HIP_CHECK_LAUNCH();
        return 0;
    }
    const bool rw1 = N <= 6144 && !paired;
    const int grid = std::min(2048, CEIL_DIV(N, rw1 ? 4 : 8));
#define GG(MV)                                                                                     \
    do {                                                                                           \
        if (rw1) hipLaunchKernelGGL((gemv_grouped_kernel<MV, 1>), dim3(grid), dim3(256), 0, s,     \
                                    (const uint32_t*)x, (const uint32_t*)w, gr, N, K / 2);         \
        else hipLaunchKernelGGL((gemv_grouped_kernel<MV, 2>), dim3(grid), dim3(256), 0, s,         \
                                (const uint32_t*)x, (const uint32_t*)w, gr, N, K / 2);             \
    } while (0)
    switch (M) {
        case 1: GG(1); break;
        case 2: GG(2); break;
        case 3: GG(3); break;
        case 4: GG(4); break;
        default: return -105;
    }
#undef GG
    HIP_CHECK_LAUNCH();
    return 0;
}
