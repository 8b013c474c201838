// Paged decode attention for MI355X (gfx950).
//
// Single new token per sequence attends to the whole paged KV cache. The op
// is HBM-bound (reads n_tokens * 2 * Hk * D * 2 bytes): 16-byte loads of cache
// rows, scores on the matrix cores, online softmax in registers, and sequences
// split over keys so that the grid covers the chip even at batch 1 (B*Hk
// workgroups alone would leave 256 CUs mostly idle).
//
// Layouts:
//   q        [B, Hq, 128] bf16
//   kc/vc    flat [num_slots, Hk, 128] bf16 (slot = block_id*block_size + off)
//   block_table [B, max_blocks] int32
//   seq_lens [B] int32 (tokens in cache, incl. the current token)
//   o_part   [B*Hk*NSPLIT, G, 128] f32, ml_part [B*Hk*NSPLIT, G, 2] f32
//   out      [B, Hq, 128] bf16
//
// A split is `chunk` keys, a multiple of 64 (decode_chunk), and at most nsplit
// splits cover a sequence; blocks past its last key end at once and the combine
// reads the splits that exist.

#include "common.h"

#define DHEAD 128

typedef __attribute__((ext_vector_type(8))) __bf16 da_b8;
typedef __attribute__((ext_vector_type(4))) float da_f4;

// Keys of a split: few splits of 64 keys leave the chip idle, many of them pay the
// per-block latency (tables, partial results) over and over. `base` comes from
// the launch (decode_chunk_base).
__device__ __forceinline__ int decode_chunk(int n, int nsplit, int base) {
    const int c = (CEIL_DIV(n, nsplit) + 63) & ~63;
    return c > base ? c : base;
}

// value of lane `N` of the own 16 lanes, and rotations within them
template <int N>
__device__ __forceinline__ float row_bcast(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + N, 0xf, 0xf, true));
}
template <int N>
__device__ __forceinline__ float row_ror(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + N, 0xf, 0xf, true));
}

// Scores on the matrix cores, values on the vector units, all in 32 bits.
//
// 16 keys x 128 channels go from the cache straight into A fragments of
// v_mfma_f32_16x16x32_bf16. A query is an exact sum of three bf16 numbers (its
// rotation is done in float32), which take three groups of the sixteen columns:
// four heads leave room for them, eight heads need a second product for the third
// part. A product of 16 keys thus costs 4 or 8 matrix instructions where dot
// products by lanes cost 4 heads x (32 multiply-adds + a 16-lane reduction) and
// bound the kernel (1.4 TB/s at batch 47). Adding the column groups is two
// rotations within 16 lanes; the lane of column c then keeps head c % GP and one
// key (two for eight heads) of its own 16-lane row, so a weight is one exponential
// per lane, and all four keys' weights of a row reach its lanes, which hold 8
// value channels each, by row broadcasts. Softmax weights, their sums and the
// value sums never leave float32. Each row keeps its own running maximum; rows,
// waves and splits are merged at the end.
//
// FUSED = true folds the split-combine into this launch with an in-launch split-K
// hand-off (plain-store form): each split block publishes its partial with an
// agent-scope release and bumps a ticket counter; the LAST arriver for (b, h)
// acquires, reads every split's slab and writes the final output. `cnt` must be
// zeroed before every launch. ROPE = true takes the raw projection outputs: the
// queries are rotated while they are split, the loop covers the CACHED keys
// [0, n-1), and the split that owns key n-1 rotates the new key, stores it and its
// value in the cache and starts its softmax with them. kin/vin/cs/sn/slots/kcw/vcw
// are only read when ROPE.
template <int G, bool FUSED, bool ROPE>
__global__ __launch_bounds__(256) void decode_attn_kernel(
    const uint32_t* __restrict__ q, const uint32_t* __restrict__ kc,
    const uint32_t* __restrict__ vc, const int* __restrict__ block_table,
    const int* __restrict__ seq_lens, float* __restrict__ o_part,
    float* __restrict__ ml_part, unsigned* __restrict__ cnt,
    uint32_t* __restrict__ out, int B, int Hk, int max_blocks,
    int block_shift /* log2(block_size) */, int nsplit, int chunk_base, float scale,
    int qs2 /* q batch-row stride in words */,
    const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
    const float* __restrict__ cs, const float* __restrict__ sn,
    const int* __restrict__ slots, uint32_t* __restrict__ kcw,
    uint32_t* __restrict__ vcw, int ks2, int vs2) {
    constexpr int GP = G > 4 ? 8 : 4;            // columns of one part of the queries
    constexpr int KL = GP / 4;                   // keys per lane and tile
    const int bh = blockIdx.x;
    const int b = bh / Hk;
    const int h = bh % Hk;
    const int split = blockIdx.y;
    const int Hq = Hk * G;

    const int n = seq_lens[b];
    const int chunk = decode_chunk(n, nsplit, chunk_base);
    const int kstart = split * chunk;
    if (!FUSED && kstart >= n) return;
    const int kend = min(n, kstart + chunk);
    // ROPE: the new key (index n-1) is handled from registers, not cache
    const int n_cached = ROPE ? (n - 1) : n;
    const int kend_c = min(kend, n_cached);

    const int lane = threadIdx.x & (WAVE - 1);
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int g16 = lane >> 4;   // row of 16 lanes: keys g16 * 4 .. + 3 of a tile
    const int dl = lane & 15;    // column; owns value channels dl*8 .. dl*8+7

    const int part_idx = (bh * nsplit + split);
    float* opart_row = o_part + ((size_t)part_idx * G) * DHEAD;
    float* mlpart_row = ml_part + ((size_t)part_idx * G) * 2;

    // per-wave sub-range (over CACHED keys only), whole tiles of 16
    const int span = max(kend_c - kstart, 0);
    const int wchunk = ((span + 63) >> 6) << 4;
    const int wstart = kstart + wid * wchunk;
    const int wend = min(kend_c, wstart + wchunk);
    const int nt = wend > wstart ? (wend - wstart + 15) >> 4 : 0;

    const int* btrow = block_table + (size_t)b * max_blocks;
    const int bmask = (1 << block_shift) - 1;
    auto slot_of = [&](int kk) {
        return (int64_t)btrow[kk >> block_shift] << block_shift | (kk & bmask);
    };
    // A tile starts at a multiple of 16 keys: pages of 16 and more hold it whole, and
    // its page is one scalar load, made a tile ahead of the rows it leads to (47 sequences
    // of up to 3000 tokens, both launches: 93.2 us with five lookups per lane and tile
    // before its loads, 85.7; 8 of up to 1500 21.0, 20.1). Two tiles ahead cost a wave
    // per SIMD: 92.
    auto page_of = [&](int t) { return btrow[(wstart + min(t, nt - 1) * 16) >> block_shift]; };
    uint4 kr_[2][4], vr_[2][4];
    auto load_tile = [&](int t, int page, uint4 (&kw)[4], uint4 (&vw)[4]) {
        const int k0 = wstart + t * 16;
        // keys past the end repeat the last one; their weights are zero
        const int last = wend - 1 - k0;
        int64_t ks, vs[4];
        if (block_shift >= 4) {
            const int64_t s0 = (int64_t)page << block_shift | (k0 & bmask);
            ks = s0 + min(dl, last);
#pragma unroll
            for (int i = 0; i < 4; ++i) vs[i] = s0 + min(g16 * 4 + i, last);
        } else {
            ks = slot_of(k0 + min(dl, last));
#pragma unroll
            for (int i = 0; i < 4; ++i) vs[i] = slot_of(k0 + min(g16 * 4 + i, last));
        }
        const uint32_t* kp = kc + ((size_t)ks * Hk + h) * (DHEAD / 2) + g16 * 4;
#pragma unroll
        for (int s = 0; s < 4; ++s) kw[s] = *reinterpret_cast<const uint4*>(kp + s * 16);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            vw[i] = *reinterpret_cast<const uint4*>(vc + ((size_t)vs[i] * Hk + h) * (DHEAD / 2) + dl * 4);
    };
    // Loads return in order: the queries and their angles are asked for first, so that they
    // are rotated and split while the first keys, values and the new key are under way
    const int head = dl % GP, part = dl / GP;
    const bool have = head < G;
    uint4 qw[4];
#pragma unroll
    for (int s = 0; s < 4; ++s)     // lane (column dl, channels s*32 + g16*8 .. + 7 of step s)
        qw[s] = *reinterpret_cast<const uint4*>(
            q + (size_t)b * qs2 + ((size_t)(h * G + (have ? head : 0)) * DHEAD + s * 32 + g16 * 8) / 2);
    float c8[2][8], s8[2][8];
    if (ROPE) {
        const int pos = max(n - 1, 0);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const float* crow = cs + (size_t)pos * (DHEAD / 2) + s * 32 + g16 * 8;
            const float* srow = sn + (size_t)pos * (DHEAD / 2) + s * 32 + g16 * 8;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                c8[s][j] = crow[j];
                s8[s][j] = srow[j];
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    int page = 0;
    if (nt > 0) {
        load_tile(0, page_of(0), kr_[0], vr_[0]);
        page = page_of(1);
    }
    const bool owner = ROPE && n - 1 >= kstart && n - 1 < kend && wid == 3;   // of the new key
    uint4 nk[4], nv;
    if (owner) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
            nk[s] = *reinterpret_cast<const uint4*>(
                kin + (size_t)b * ks2 + ((size_t)h * DHEAD + s * 32 + g16 * 8) / 2);
        nv = *reinterpret_cast<const uint4*>(vin + (size_t)b * vs2 + ((size_t)h * DHEAD + dl * 8) / 2);
    }
    __builtin_amdgcn_sched_barrier(0);

    float qf[4][8];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            qf[s][j * 2] = have ? bf16_lo((&qw[s].x)[j]) : 0.0f;
            qf[s][j * 2 + 1] = have ? bf16_hi((&qw[s].x)[j]) : 0.0f;
        }
    // ROPE: channel d pairs with d + 64, two steps on in the same lane
    if (ROPE) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float x1 = qf[s][j], x2 = qf[s + 2][j];
                qf[s][j] = x1 * c8[s][j] - x2 * s8[s][j];
                qf[s + 2][j] = x2 * c8[s][j] + x1 * s8[s][j];
            }
    }

    // the lane's part of its query, and the third parts for a second product: the first
    // bf16 of what the parts before leave
    da_b8 qb[4], qb2[GP == 8 ? 4 : 1];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float x = qf[s][j], hi = (float)(__bf16)x;
            if (GP == 8) {
                const float r1 = x - hi, mid = (float)(__bf16)r1;
                qb[s][j] = (__bf16)(part == 0 ? x : r1);
                qb2[GP == 8 ? s : 0][j] = (__bf16)(part == 0 ? r1 - mid : 0.0f);
            } else {
                const float r1 = part > 0 ? x - hi : x;
                const float r2 = part > 1 ? r1 - (float)(__bf16)r1 : r1;
                qb[s][j] = (__bf16)(part < 3 ? r2 : 0.0f);
            }
        }

    // running maximum of the lane's head over its row's keys, the lane's share of
    // the sum of weights, value sums of all heads
    float m = -INFINITY, lsum = 0.0f, o[G][8];
#pragma unroll
    for (int gh = 0; gh < G; ++gh)
#pragma unroll
        for (int j = 0; j < 8; ++j) o[gh][j] = 0.0f;

    if (owner) {
        float kf[4][8];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                kf[s][j * 2] = bf16_lo((&nk[s].x)[j]);
                kf[s][j * 2 + 1] = bf16_hi((&nk[s].x)[j]);
            }
        float dot = 0.0f;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float x1 = kf[s][j], x2 = kf[s + 2][j];
                kf[s][j] = x1 * c8[s][j] - x2 * s8[s][j];
                kf[s + 2][j] = x2 * c8[s][j] + x1 * s8[s][j];
                dot = fmaf(qf[s][j], kf[s][j], dot);
                dot = fmaf(qf[s + 2][j], kf[s + 2][j], dot);
            }
        dot += __shfl_xor(dot, 16, WAVE);
        dot += __shfl_xor(dot, 32, WAVE);
        const int64_t slot = slots[b];
        if (dl == 0) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
                *reinterpret_cast<uint4*>(kcw + ((size_t)slot * Hk + h) * (DHEAD / 2) + s * 16 + g16 * 4) =
                    make_uint4(pack_bf16x2(kf[s][0], kf[s][1]), pack_bf16x2(kf[s][2], kf[s][3]),
                               pack_bf16x2(kf[s][4], kf[s][5]), pack_bf16x2(kf[s][6], kf[s][7]));
        }
        if (g16 == 0) {
            *reinterpret_cast<uint4*>(vcw + ((size_t)slot * Hk + h) * (DHEAD / 2) + dl * 4) = nv;
            m = dot * scale;
            lsum = part == 0 ? 1.0f : 0.0f;
#pragma unroll
            for (int gh = 0; gh < G; ++gh)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    o[gh][j * 2] = bf16_lo((&nv.x)[j]);
                    o[gh][j * 2 + 1] = bf16_hi((&nv.x)[j]);
                }
        }
    }

    auto process = [&](int t, const uint4 (&kw)[4], const uint4 (&vw)[4]) {
        da_f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 4; ++s)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(da_b8, kw[s]), qb[s], acc, 0, 0, 0);
        if (GP == 8) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(da_b8, kw[s]),
                                                              qb2[GP == 8 ? s : 0], acc, 0, 0, 0);
        }
        float x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[i] = acc[i];
            if (GP == 4) x[i] += row_ror<4>(x[i]);
            x[i] += row_ror<8>(x[i]);
        }
        // An infinite key times a part that is zero is NaN: such a key's score is that of the
        // first parts alone, infinite or NaN as the whole query's is
        const float xs = (x[0] + x[1]) + (x[2] + x[3]);
        if (__any(xs != xs)) {
            da_f4 first = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < 4; ++s)
                first = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(da_b8, kw[s]), qb[s], first, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float y = __shfl(first[i], (lane & 48) | head, WAVE);
                if (x[i] != x[i]) x[i] = y;
            }
        }
        // the lane's own keys of its row
        float sc[KL], p[KL];
        const int key = wstart + t * 16 + g16 * 4 + part * KL;
        if (GP == 4) {
            sc[0] = part & 2 ? (part & 1 ? x[3] : x[2]) : (part & 1 ? x[1] : x[0]);
        } else {
            sc[0] = part ? x[2] : x[0];
            sc[KL - 1] = part ? x[3] : x[1];
        }
        float mx = m;
#pragma unroll
        for (int i = 0; i < KL; ++i) {
            sc[i] = key + i < wend ? sc[i] * scale : -INFINITY;
            mx = fmaxf(mx, sc[i]);
        }
        if (GP == 4) mx = fmaxf(mx, row_ror<4>(mx));
        mx = fmaxf(mx, row_ror<8>(mx));
        const float ref = mx == -INFINITY ? 0.0f : mx;
        const float alpha = __expf(m - ref);
        m = mx;
        lsum *= alpha;
#pragma unroll
        for (int i = 0; i < KL; ++i) {
            p[i] = __expf(sc[i] - ref);
            lsum += p[i];
        }
        // rescale the value sums only where some row's maximum moved
        if (__any(alpha != 1.0f)) {
            float al[8];
            al[0] = row_bcast<0>(alpha); al[1] = row_bcast<1>(alpha);
            al[2] = row_bcast<2>(alpha); al[3] = row_bcast<3>(alpha);
            al[4] = row_bcast<4>(alpha); al[5] = row_bcast<5>(alpha);
            al[6] = row_bcast<6>(alpha); al[7] = row_bcast<7>(alpha);
#pragma unroll
            for (int gh = 0; gh < G; ++gh)
#pragma unroll
                for (int j = 0; j < 8; ++j) o[gh][j] *= al[gh];
        }
#define DA_KEY(I)                                                                              \
    {                                                                                          \
        float vf[8], pb[8];                                                                    \
        _Pragma("unroll") for (int j = 0; j < 4; ++j) {                                        \
            vf[j * 2] = bf16_lo((&vw[I].x)[j]);                                                \
            vf[j * 2 + 1] = bf16_hi((&vw[I].x)[j]);                                            \
        }                                                                                      \
        const float pv = p[GP == 4 ? 0 : ((I) & 1)];                                           \
        constexpr int c0 = GP == 4 ? (I) * 4 : ((I) >> 1) * 8;                                 \
        pb[0] = row_bcast<c0 + 0>(pv);                                                         \
        if (G > 1) pb[1] = row_bcast<c0 + 1>(pv);                                              \
        if (G > 2) {                                                                           \
            pb[2] = row_bcast<c0 + 2>(pv);                                                     \
            pb[3] = row_bcast<c0 + 3>(pv);                                                     \
        }                                                                                      \
        if (G > 4) {                                                                           \
            pb[4] = row_bcast<(c0 + 4) & 15>(pv);                                              \
            pb[5] = row_bcast<(c0 + 5) & 15>(pv);                                              \
            pb[6] = row_bcast<(c0 + 6) & 15>(pv);                                              \
            pb[7] = row_bcast<(c0 + 7) & 15>(pv);                                              \
        }                                                                                      \
        _Pragma("unroll") for (int gh = 0; gh < G; ++gh)                                       \
            _Pragma("unroll") for (int j = 0; j < 8; ++j)                                      \
                o[gh][j] = fmaf(pb[gh], vf[j], o[gh][j]);                                      \
    }
        DA_KEY(0) DA_KEY(1) DA_KEY(2) DA_KEY(3)
#undef DA_KEY
    };
    // one tile in flight behind the one in work; the last load repeats its tile, so
    // that waits count exactly
    for (int t = 0; t < nt; t += 2) {
        load_tile(min(t + 1, nt - 1), page, kr_[1], vr_[1]);
        page = page_of(t + 2);
        __builtin_amdgcn_sched_barrier(0);
        process(t, kr_[0], vr_[0]);
        if (t + 1 < nt) {
            load_tile(min(t + 2, nt - 1), page, kr_[0], vr_[0]);
            page = page_of(t + 3);
            __builtin_amdgcn_sched_barrier(0);
            process(t + 1, kr_[1], vr_[1]);
        }
    }

    // sums and maxima of every head to all lanes of a row
    if (GP == 4) lsum += row_ror<4>(lsum);
    lsum += row_ror<8>(lsum);
    float mh[8], lh[8];
    mh[0] = row_bcast<0>(m); mh[1] = row_bcast<1>(m); mh[2] = row_bcast<2>(m); mh[3] = row_bcast<3>(m);
    mh[4] = row_bcast<4>(m); mh[5] = row_bcast<5>(m); mh[6] = row_bcast<6>(m); mh[7] = row_bcast<7>(m);
    lh[0] = row_bcast<0>(lsum); lh[1] = row_bcast<1>(lsum); lh[2] = row_bcast<2>(lsum); lh[3] = row_bcast<3>(lsum);
    lh[4] = row_bcast<4>(lsum); lh[5] = row_bcast<5>(lsum); lh[6] = row_bcast<6>(lsum); lh[7] = row_bcast<7>(lsum);

    // merge the wave's 4 key-groups (lanes l, l^16, l^32 hold same dims)
#pragma unroll
    for (int off = 16; off <= 32; off <<= 1) {
#pragma unroll
        for (int gh = 0; gh < G; ++gh) {
            const float m2 = __shfl_xor(mh[gh], off, WAVE);
            const float l2 = __shfl_xor(lh[gh], off, WAVE);
            float o2[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) o2[j] = __shfl_xor(o[gh][j], off, WAVE);
            const float mn = fmaxf(mh[gh], m2);
            // guard: empty partial (l == 0, m == -inf) must not produce NaN
            const float a1 = (lh[gh] > 0.0f) ? __expf(mh[gh] - mn) : 0.0f;
            const float a2 = (l2 > 0.0f) ? __expf(m2 - mn) : 0.0f;
#pragma unroll
            for (int j = 0; j < 8; ++j) o[gh][j] = o[gh][j] * a1 + o2[j] * a2;
            lh[gh] = lh[gh] * a1 + l2 * a2;
            mh[gh] = (lh[gh] > 0.0f) ? mn : -INFINITY;
        }
    }

    // cross-wave combine through LDS
    __shared__ float lds_o[4][G][DHEAD];
    __shared__ float lds_ml[4][G][2];
    if (lane < 16) {
#pragma unroll
        for (int gh = 0; gh < G; ++gh) {
#pragma unroll
            for (int j = 0; j < 8; ++j) lds_o[wid][gh][dl * 8 + j] = o[gh][j];
            if (dl == 0) {
                lds_ml[wid][gh][0] = mh[gh];
                lds_ml[wid][gh][1] = lh[gh];
            }
        }
    }
    __syncthreads();

    // 256 threads cover G*128 outputs
    for (int idx = threadIdx.x; idx < G * DHEAD; idx += blockDim.x) {
        const int gh = idx / DHEAD;
        const int d = idx % DHEAD;
        float mt = -INFINITY;
#pragma unroll
        for (int w = 0; w < 4; ++w)
            if (lds_ml[w][gh][1] > 0.0f) mt = fmaxf(mt, lds_ml[w][gh][0]);
        float lt = 0.0f, ot = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float lw = lds_ml[w][gh][1];
            if (lw > 0.0f) {
                const float sc = __expf(lds_ml[w][gh][0] - mt);
                lt += lw * sc;
                ot += lds_o[w][gh][d] * sc;
            }
        }
        opart_row[gh * DHEAD + d] = ot;
        if (d == 0) {
            mlpart_row[gh * 2 + 0] = mt;
            mlpart_row[gh * 2 + 1] = lt;
        }
    }

    if (!FUSED) return;

    // ---- G16 publish + reducer election (plain-store recipe) --------------
    // every wave drains its slab stores, then one lane releases and takes a
    // ticket; the block that draws nsplit-1 becomes the reducer
    __shared__ int s_last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // EVERY wave
    __syncthreads();
    if (threadIdx.x == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        // restate the post-wbl2 wait the compiler may drop (guide pitfall 12)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const unsigned prev = __hip_atomic_fetch_add(
            &cnt[bh], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = (prev == (unsigned)(nsplit - 1));
    }
    __syncthreads();
    if (!s_last) return;
    if (threadIdx.x == 0)
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // drop stale L1
    __syncthreads();

    // ---- reduce all splits of (b, h) and write the final O ----------------
    const int Hq2 = Hk * G;
    const int base = bh * nsplit;
    for (int idx = threadIdx.x; idx < G * DHEAD; idx += blockDim.x) {
        const int gh = idx / DHEAD;
        const int d = idx % DHEAD;
        float mt = -INFINITY;
        for (int s = 0; s < nsplit; ++s) {
            const float lw = ml_part[((size_t)(base + s) * G + gh) * 2 + 1];
            if (lw > 0.0f) mt = fmaxf(mt, ml_part[((size_t)(base + s) * G + gh) * 2]);
        }
        float lt = 0.0f, ot = 0.0f;
        for (int s = 0; s < nsplit; ++s) {
            const float mw = ml_part[((size_t)(base + s) * G + gh) * 2];
            const float lw = ml_part[((size_t)(base + s) * G + gh) * 2 + 1];
            if (lw > 0.0f) {
                const float sc = __expf(mw - mt);
                lt += lw * sc;
                ot += o_part[((size_t)(base + s) * G + gh) * DHEAD + d] * sc;
            }
        }
        const float res = (lt > 0.0f) ? ot / lt : 0.0f;
        reinterpret_cast<uint16_t*>(out)[(size_t)(b * Hq2 + h * G + gh) * DHEAD + d] =
            f32_to_bf16(res);
    }
}

// Combine split partials -> final output. Grid: B*Hq blocks, 512 threads:
// thread (d = tid & 127, sh = tid >> 7) accumulates splits sh, sh+4, ... so
// the split loop runs nsplit/4 iterations with 4-way ILP, then the 4 partial
// (m, l, o_d) triples merge through LDS. The (m, l) table is staged into LDS
// once by the first wave (the naive one-thread-one-d loop over 64 splits was
// 32 us/launch — 3x the attention kernel itself).
template <int G>
__global__ __launch_bounds__(512) void decode_combine_kernel(
    const float* __restrict__ o_part, const float* __restrict__ ml_part,
    const int* __restrict__ seq_lens, uint32_t* __restrict__ out, int B, int Hk, int nsplit,
    int chunk_base) {
    const int bq = blockIdx.x;
    const int Hq = Hk * G;
    const int b = bq / Hq;
    const int qh = bq % Hq;
    const int h = qh / G;
    const int gh = qh % G;
    const int d = threadIdx.x & (DHEAD - 1);
    const int sh = threadIdx.x >> 7;  // 0..3

    extern __shared__ __attribute__((aligned(16))) float sml[];  // [nsplit][2]
    const int base = (b * Hk + h) * nsplit;
    const int n = seq_lens[b];
    const int ns = CEIL_DIV(n, decode_chunk(n, nsplit, chunk_base));
    for (int s = threadIdx.x; s < ns; s += blockDim.x) {
        const float2 ml = *reinterpret_cast<const float2*>(
            ml_part + ((size_t)(base + s) * G + gh) * 2);
        sml[s * 2] = ml.x;
        sml[s * 2 + 1] = ml.y;
    }
    __syncthreads();

    float mt = -INFINITY;
    for (int s = sh; s < ns; s += 4)
        if (sml[s * 2 + 1] > 0.0f) mt = fmaxf(mt, sml[s * 2]);
    float lt = 0.0f, ot = 0.0f;
    for (int s = sh; s < ns; s += 4) {
        const float lw = sml[s * 2 + 1];
        if (lw > 0.0f) {
            const float sc = __expf(sml[s * 2] - mt);
            lt += lw * sc;
            ot += o_part[((size_t)(base + s) * G + gh) * DHEAD + d] * sc;
        }
    }
    // merge the 4 split-groups via LDS (per d): (m, l, o) online combine
    __shared__ float red_m[4][DHEAD], red_l[4][DHEAD], red_o[4][DHEAD];
    red_m[sh][d] = mt;
    red_l[sh][d] = lt;
    red_o[sh][d] = ot;
    __syncthreads();
    if (sh == 0) {
#pragma unroll
        for (int g2 = 1; g2 < 4; ++g2) {
            const float m2 = red_m[g2][d], l2 = red_l[g2][d], o2 = red_o[g2][d];
            const float mn = fmaxf(mt, m2);
            const float a1 = (lt > 0.0f) ? __expf(mt - mn) : 0.0f;
            const float a2 = (l2 > 0.0f) ? __expf(m2 - mn) : 0.0f;
            ot = ot * a1 + o2 * a2;
            lt = lt * a1 + l2 * a2;
            mt = (lt > 0.0f) ? mn : -INFINITY;
        }
        const float res = (lt > 0.0f) ? ot / lt : 0.0f;
        reinterpret_cast<uint16_t*>(out)[(size_t)(b * Hq + qh) * DHEAD + d] =
            f32_to_bf16(res);
    }
}

// Keys of the smallest split, by the (sequence, key head) pairs of the launch. Both
// launches, 8 key heads, us with 64 / 128 / 256 / 512 keys: one sequence of 1151
// tokens 14.4 / 14.5 / 15.9 / 19.3 (16.8 before scores ran on the matrix cores),
// 8 of up to 1500 29.3 / 20.6 / 20.6 / 21.2 (38.5), 16 43.3 / 32.0 / 27.8 / 30.4
// (64.3), 32 of up to 3000 104 / 86 / 72 / 69 (146), 64 180 / 153 / 129 / 117 (266;
// its cache rows alone take 89 at 5.5 TB/s), 64 of up to 300 39 / 31 / 27 / 26 (152).
static int decode_chunk_base(int pairs) {
    return pairs <= 8 ? 64 : pairs <= 64 ? 128 : pairs <= 128 ? 256 : 512;
}

// fused: cnt_ws is zeroed here on each call (hipMemsetAsync). fused = 0: two kernels.
extern "C" int oa_attention_decode(void* stream, const void* q, const void* kc,
                                   const void* vc, const void* block_table,
                                   const void* seq_lens, void* o_part,
                                   void* ml_part, void* cnt_ws, void* out, int B,
                                   int Hq, int Hk, int D, int max_blocks,
                                   int block_size, int nsplit, float scale,
                                   int q_stride, int fused) {
    if (q_stride % 8 != 0) return -103;
    const int qs2 = q_stride / 2;
    if (D != DHEAD) return -100;
    if ((block_size & (block_size - 1)) != 0) return -101;
    const int G = Hq / Hk;
    int block_shift = 0;
    while ((1 << block_shift) < block_size) ++block_shift;
    dim3 grid(B * Hk, nsplit), block(256);
    dim3 cgrid(B * Hq), cblock(512);
    const int clds = nsplit * 2 * (int)sizeof(float);

    if (fused) {
        hipError_t e = hipMemsetAsync(cnt_ws, 0, B * Hk * 4, (hipStream_t)stream);
        if (e != hipSuccess) return (int)e;
    }

    const int cb = decode_chunk_base(B * Hk);
#define LAUNCH_G(GV)                                                                \
    do {                                                                            \
        if (fused) {                                                                \
            hipLaunchKernelGGL((decode_attn_kernel<GV, true, false>), grid, block,         \
                               0, (hipStream_t)stream, (const uint32_t*)q,          \
                               (const uint32_t*)kc, (const uint32_t*)vc,            \
                               (const int*)block_table, (const int*)seq_lens,       \
                               (float*)o_part, (float*)ml_part, (unsigned*)cnt_ws,  \
                               (uint32_t*)out, B, Hk, max_blocks, block_shift,      \
                               nsplit, cb, scale, qs2, (const uint32_t*)nullptr,        \
                               (const uint32_t*)nullptr, (const float*)nullptr,     \
                               (const float*)nullptr, (const int*)nullptr,          \
                               (uint32_t*)nullptr, (uint32_t*)nullptr, 0, 0);       \
            HIP_CHECK_LAUNCH();                                                     \
        } else {                                                                    \
            hipLaunchKernelGGL((decode_attn_kernel<GV, false, false>), grid, block,        \
                               0, (hipStream_t)stream, (const uint32_t*)q,          \
                               (const uint32_t*)kc, (const uint32_t*)vc,            \
                               (const int*)block_table, (const int*)seq_lens,       \
                               (float*)o_part, (float*)ml_part, (unsigned*)cnt_ws,  \
                               (uint32_t*)out, B, Hk, max_blocks, block_shift,      \
                               nsplit, cb, scale, qs2, (const uint32_t*)nullptr,        \
                               (const uint32_t*)nullptr, (const float*)nullptr,     \
                               (const float*)nullptr, (const int*)nullptr,          \
                               (uint32_t*)nullptr, (uint32_t*)nullptr, 0, 0);       \
            HIP_CHECK_LAUNCH();                                                     \
            hipLaunchKernelGGL((decode_combine_kernel<GV>), cgrid, cblock, clds,    \
                               (hipStream_t)stream, (const float*)o_part,           \
                               (const float*)ml_part, (const int*)seq_lens,         \
                               (uint32_t*)out, B, Hk, nsplit, cb);                                             \
            HIP_CHECK_LAUNCH();                                                     \
        }                                                                           \
    } while (0)

    switch (G) {
        case 1: LAUNCH_G(1); break;
        case 2: LAUNCH_G(2); break;
        case 4: LAUNCH_G(4); break;
        case 8: LAUNCH_G(8); break;
        default: return -102;
    }
#undef LAUNCH_G
    return 0;
}

// Fully-fused decode attention: RoPE(q, k) + paged-KV scatter of (k, v) +
// split-K attention in ONE launch (+ the combine kernel) — replaces the
// separate rope_kv launch per layer. q/kin/vin are the RAW (un-roped) GEMV
// outputs; kc/vc are read for cached keys and written at slots[b].
extern "C" int oa_attention_decode_rope(
    void* stream, const void* q, const void* kin, const void* vin, void* kc,
    void* vc, const void* block_table, const void* seq_lens, const void* cos_t,
    const void* sin_t, const void* slots, void* o_part, void* ml_part,
    void* out, int B, int Hq, int Hk, int D, int max_blocks, int block_size,
    int nsplit, float scale, int q_stride, int k_stride, int v_stride) {
    if ((q_stride | k_stride | v_stride) % 8 != 0) return -103;
    if (D != DHEAD) return -100;
    if ((block_size & (block_size - 1)) != 0) return -101;
    const int G = Hq / Hk;
    int block_shift = 0;
    while ((1 << block_shift) < block_size) ++block_shift;
    dim3 grid(B * Hk, nsplit), block(256);
    dim3 cgrid(B * Hq), cblock(512);
    const int clds = nsplit * 2 * (int)sizeof(float);

    const int cb = decode_chunk_base(B * Hk);
#define LAUNCH_GR(GV)                                                              \
    do {                                                                            \
        hipLaunchKernelGGL((decode_attn_kernel<GV, false, true>), grid, block, 0,   \
                           (hipStream_t)stream, (const uint32_t*)q,                 \
                           (const uint32_t*)kc, (const uint32_t*)vc,                \
                           (const int*)block_table, (const int*)seq_lens,           \
                           (float*)o_part, (float*)ml_part, (unsigned*)nullptr,     \
                           (uint32_t*)out, B, Hk, max_blocks, block_shift, nsplit,  \
                           cb, scale, q_stride / 2, (const uint32_t*)kin,               \
                           (const uint32_t*)vin, (const float*)cos_t,               \
                           (const float*)sin_t, (const int*)slots, (uint32_t*)kc,   \
                           (uint32_t*)vc, k_stride / 2, v_stride / 2);              \
        HIP_CHECK_LAUNCH();                                                         \
        hipLaunchKernelGGL((decode_combine_kernel<GV>), cgrid, cblock, clds,        \
                           (hipStream_t)stream, (const float*)o_part,               \
                           (const float*)ml_part, (const int*)seq_lens,             \
                           (uint32_t*)out, B, Hk, nsplit, cb);                      \
        HIP_CHECK_LAUNCH();                                                         \
    } while (0)

    switch (G) {
        case 1: LAUNCH_GR(1); break;
        case 2: LAUNCH_GR(2); break;
        case 4: LAUNCH_GR(4); break;
        case 8: LAUNCH_GR(8); break;
        default: return -102;
    }
#undef LAUNCH_GR
    return 0;
}
