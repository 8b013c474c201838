// Flash-style causal prefill attention for MI355X (gfx950): bf16 matrix instructions, K and V
// staged through LDS, softmax in registers.
//
//   * K AND V staged by transfers into LDS (16-B pieces) in a 2-deep ring: tile t+1's
//     transfers are in flight under tile t's compute
//   * K image: 256-B key rows, XOR swizzle byte^=(key&15)<<4 applied on
//     the transfer's SOURCE address (the LDS write is
//     lane-linear, so the swizzle moves to the per-lane global address)
//     and on the ds_read_b128 A-fragment reads
//   * V image: [KB/32 key blocks][8 d-block] subtiles of [32 key][16 d] bf16
//     with key bits permuted (img_row = (k&3) + ((k>>3)<<2) + ((k&4)<<2))
//     so each ds_read_b64_tr_b16 serves the P·V fragment conflict-free
//   * a wave owns 32 q-rows; lane's l&31 IS its q-row, so softmax stats are
//     per-lane scalars and each row reduction is ONE exchange with lane^32
//   * S^T = mfma(A=K, B=Q): C[row=key][col=q-row] puts half of a tile's scores of a
//     lane's row (partner lane l^32 holds the other half) in 32x32 accumulators,
//     masked and softmaxed in registers
//   * P -> P·V operand WITHOUT an LDS round-trip: score quads packed to
//     bf16 pairs, one half exchanged with the partner lane, and
//     O^T = mfma(A=V^T, B=P^T) keeps the lane<->q-row mapping (alpha rescale
//     stays a per-lane scalar multiply)
//   * per-tile wave-uniform branches skip masking on fully-unmasked tiles
//     and skip compute entirely on tiles past the wave's causal diagonal
//
// What bounds it: with two waves a SIMD the matrix instructions (4096 cycles for 256 rows x
// 128 keys, 1.7 us) and about as many cycles of vector instructions hardly overlap, and a
// tile takes 4.2 us. So the time of a launch is the longest chain of tiles on one CU, and
// the split of the work is about chains:
//   * Key groups (KG): 8 waves as one group of 256 rows, two of 128 or four of 64, each group
//     on its own tiles of the keys, summed up in LDS at the end. 128 keys take 4.2, 2.6 and
//     2.0 us: the chip's rate falls, but so do a short prompt's chains, with the same blocks.
//   * Longest chains first (causal prompts have blocks of one to many tiles): late blocks fill
//     up the CUs that are done, and the heads of a key head are a multiple of 8 blocks apart
//     (8 key heads), that is on one XCD, whose L2 then holds their keys.
// us, 32 heads on 8, before both / now: 800 queries of 1024 keys 41.7 / 27.2, 700 of 700
// 27.4 / 19.2, 1434 of 1434 53 / 34.4, 2048 of 2048 74 / 53.6, 4096 of 4096 250 / 153, 2048 of
// 6144 201 / 199; 16 on 4, 512 of 512 19.1 / 13.2; split, 77 of 1187 26 / 17.
//
// Out-of-range keys are CLAMPED to Skv-1 on the transfer source and their
// scores masked to -inf (P=0 nullifies the garbage V contribution), so
// partial tail tiles need no separate path.
//
// Layouts: q [B, Sq, Hq, 128], k/v [B, Skv, Hk, 128] with per-token strides
// (they may be head-slices of one fused qkv buffer), out [B, Sq, Hq, 128]
// contiguous; causal offset = Skv - Sq (query i attends keys [0..Skv-Sq+i])
// so multi-turn chunked prefill reuses the same kernel. With `slots` (int64 [Skv], one
// sequence) key i is row slots[i] of the `rows` that k and v have, the cache's as they lie.

#include "common.h"

#define DHEAD 128
#define NWAVE 8

typedef __attribute__((ext_vector_type(8))) short bf16x8_t;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4v;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;

__device__ __forceinline__ uint32_t k_swz_read(int key, int byte_in_row) {
    return (uint32_t)(key * (DHEAD * 2) + (byte_in_row ^ ((key & 15) << 4)));
}

// V image row permutation: key -> subtile row (see header)
__device__ __forceinline__ int v_img_row_inv(int r) {
    // inverse: img_row r -> key
    return (r & 3) + (((r >> 4) & 1) << 2) + (((r >> 2) & 3) << 3);
}

// Partner-half (lane ^ 32) value on the VALU: v_permlane32_swap with equal
// inputs yields r[0] = [lo|lo], r[1] = [hi|hi], so the partner's value is
// r[1] for the low half and r[0] for the high half. The two-asm-operand
// form is NOT equivalent (measured on-box: the upper half saw its own
// value) — the builtin models both register updates correctly.
__device__ __forceinline__ float xor32_f32(float v, int lh) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(lh ? r[0] : r[1]);
}

// The row that an entry of `slots` names, by its low word: one below 0 counts from the end, as an index
// of a tensor does, and what lies outside either way reads the last row, not what is beside the cache.
// Two instructions (unsigned, slot + rows is the larger one but below 0); with all 64 bits compared
// 2048 queries of 6144 keys took 4% longer.
__device__ __forceinline__ int cache_row(int slot, int rows) {
    return (int)min(min((uint32_t)slot, (uint32_t)slot + (uint32_t)rows), (uint32_t)(rows - 1));
}

// PAGED: the blocks of a key head, which share an XCD's L2, ask for up to four lines a lane of
// all its keys and values while the first tile is under way: cache rows come from memory, and a
// step of 1 to 2 us is less than its latency. `me` of `sharers` blocks; the caller waits. Four
// layers of a model, us, gathered / from the cache / so: 600 behind 1800, 32 heads on 8, 1430 / 1458 /
// 1426; 1500 tokens behind 3000, 16 on 4, 1222 / 1300 / 1242, of the few that stay behind a gather (1500
// behind 6000 1530 / - / 1562).
constexpr int TOUCHES = 4;
__device__ __forceinline__ void touch_rows(uint32_t (&t)[TOUCHES], const char* kbase, const char* vbase,
                                           const int64_t* slots, int rows, int64_t kstep, int64_t vstep,
                                           int key0, int key1, int me, int sharers) {
#pragma unroll
    for (int i = 0; i < TOUCHES; ++i) {
        const int line = min((i * sharers + me) * 512 + (int)threadIdx.x, 4 * (key1 - key0) - 1);
        const int row = cache_row(reinterpret_cast<const int*>(slots)[2 * (key0 + (line >> 2))], rows);
        const char* at = line & 2 ? vbase + row * vstep : kbase + row * kstep;
        t[i] = *reinterpret_cast<const uint32_t*>(at + (line & 1) * 128);
    }
}

// GQ > 1: the workgroup carries GQ q-heads that SHARE one KV head
// (requires Hq/Hk == GQ): waves split into GQ sets, each owning QTILE/GQ q-rows of its head,
// and every staged K/V tile feeds all of them (2 to 4 per cent over a block per head).
// SPLIT: blockIdx.z takes a run of the q-tile's key tiles and leaves its unnormalised
// float32 sums with their maximum (raw scores) and weight sum for
// prefill_combine_kernel: few queries over many keys fill the chip this way.
template <int KG, int GQ, bool SPLIT, bool PAGED>
__global__ __launch_bounds__(512, 1) void attn_prefill_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
    const uint16_t* __restrict__ v, uint16_t* __restrict__ out, int B, int Hq,
    int Hk, int Sq, int Skv, float scale, int qs, int ks, int vs,
    float* __restrict__ po, float* __restrict__ pml, const int64_t* __restrict__ slots, int rows) {
    constexpr int KB = 128 / KG;             // keys of a group's tile: 128 of LDS' 160 KiB
    constexpr int QROWS = 32;                // per wave
    constexpr int NG = NWAVE / KG;           // waves of a key group
    constexpr int QTILE = QROWS * NG;        // 256 / KG across the WG
    constexpr int QTILE_H = QTILE / GQ;      // rows per head per WG
    constexpr int KBYTES = KB * DHEAD * 2;   // one K (or V) ring buffer
    constexpr int PIECES = KB / (4 * NG);    // 1-KiB DMA chunks per wave
    constexpr int NKB32 = KB / 32;           // 32-key score blocks
    __shared__ __attribute__((aligned(16))) char lds[4 * KBYTES * KG];
    const uint32_t voff = 2 * KBYTES;        // V buffers after the K ring

    // longest chains first; the heads of a key head B * Hk blocks apart
    const int groups = Hq / Hk / GQ, pairs = B * Hk, nbh = pairs * groups;
    const int turn = blockIdx.x / nbh, place = blockIdx.x % nbh;
    const int qtile = CEIL_DIV(Sq, QTILE_H) - 1 - turn;
    const int bh = place % pairs * groups + place / pairs;   // spans B * (Hq/GQ)
    const int tid = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int gid = KG > 1 ? __builtin_amdgcn_readfirstlane(tid / (WAVE * NG)) : 0;
    const int wid = tid / WAVE - gid * NG;   // within the key group
    char* const smem = lds + gid * 4 * KBYTES;
    const int b = bh / (Hq / GQ);
    const int h = (bh % (Hq / GQ)) * GQ + wid / (NG / GQ);
    const int hk = h / (Hq / Hk);
    const int offset = Skv - Sq;

    const int l31 = lane & 31;  // the lane's q-row within the wave block
    const int lh = lane >> 5;   // fragment k-half (and score key-quad offset)

    // ---- Q: B-fragment per d-step s: bq[s] = Q[row l31][d = s*16 + lh*8 ..+7]
    const int qrow0 = qtile * QTILE_H + (wid % (NG / GQ)) * QROWS;
    const int qrow = qrow0 + l31;
    uint4 bq[8];
    if (qrow < Sq) {
        const uint16_t* qp = q + (size_t)(b * Sq + qrow) * qs + (size_t)h * DHEAD;
#pragma unroll
        for (int s = 0; s < 8; ++s)
            bq[s] = *reinterpret_cast<const uint4*>(qp + s * 16 + lh * 8);
    } else {
#pragma unroll
        for (int s = 0; s < 8; ++s) bq[s] = make_uint4(0, 0, 0, 0);
    }

    float m = -INFINITY, lsum = 0.0f;
    f32x16_t oa[4];
#pragma unroll
    for (int db = 0; db < 4; ++db) oa[db] = (f32x16_t)(0.0f);

    const int kv_needed = min(Skv, offset + qtile * QTILE_H + QTILE_H);
    const int all_tiles = CEIL_DIV(max(kv_needed, 0), KB);
    const int run = SPLIT ? CEIL_DIV(all_tiles, (int)gridDim.z) : all_tiles;
    const int tile0 = SPLIT ? (int)blockIdx.z * run : 0;
    const int ntiles = SPLIT ? min(all_tiles, tile0 + run) : all_tiles;

    const char* kbase = reinterpret_cast<const char*>(k) +
                        ((size_t)b * Skv * ks + (size_t)hk * DHEAD) * 2;
    const char* vbase = reinterpret_cast<const char*>(v) +
                        ((size_t)b * Skv * vs + (size_t)hk * DHEAD) * 2;
    const int skv_clamp = Skv - 1;

    // The transfers are issued by INLINE ASM, not the builtin: hipcc's machine-
    // level wait inserter cannot disambiguate a runtime LDS destination
    // from the compute phase's ds_reads and drains the ring with a vmcnt(0)
    // before the first ds_read of every tile, which serializes the whole
    // pipeline (measured in the assembly for both builtin forms). Untracked asm
    // transfers leave wait placement to us: one explicit vmcnt(0) right before
    // each tile barrier, so tile t+1's transfers stream under tile t's MFMAs.
    // (Untracked VMEM only ever makes the compiler's own counted waits
    // MORE conservative, as vmcnt retires in issue order, never unsafe.)
    //
    // EVERY asm operand is a LOOP-PERSISTENT value updated only at the loop
    // top: the wait inserter marks asm operands as pending defs, so if a
    // compute-phase instruction reuses one of those registers it inserts a
    // drain mid-compute. Persistent
    // operands pin the registers for the whole loop; the only inserted
    // waits land right after our own vmcnt(0), where they are free.
    // a wave's pieces of V are channels of the same keys
    int k_byte[PIECES], v_byte[PIECES], kkey0[PIECES], vkey0 = 0;
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
        const int c = wid * PIECES + p;
        const int kkey = c * 4 + (lane >> 4);
        kkey0[p] = kkey;
        k_byte[p] = ((lane & 15) * 16) ^ ((kkey & 15) << 4);
        const int kb2 = c >> 3, nb = c & 7;
        vkey0 = kb2 * 32 + v_img_row_inv(lane >> 1);
        v_byte[p] = (nb * 16 + (lane & 1) * 8) * 2;
    }
    uint32_t m0k[2][PIECES], m0v[2][PIECES];
#pragma unroll
    for (int buf = 0; buf < 2; ++buf)
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            const int c = wid * PIECES + p;
            m0k[buf][p] = __builtin_amdgcn_readfirstlane(
                (uint32_t)(uintptr_t)smem + buf * KBYTES + c * 1024);
            m0v[buf][p] = __builtin_amdgcn_readfirstlane(
                (uint32_t)(uintptr_t)smem + voff + buf * KBYTES + c * 1024);
        }
    const char* ksrc[PIECES];
    const char* vsrc[PIECES];
    uint32_t m0k_cur[PIECES], m0v_cur[PIECES];
    // PAGED: the rows of a tile are looked up a tile ahead of its transfers, straight-line and
    // as loaded, so that the only wait for them is the drain
    int krow[PIECES], vrow = 0;
    auto find_rows = [&](int t) {
        const int kv0 = t * KB;
        auto row = [&](int key) {
            const int at = min(kv0 + key, skv_clamp);
            return PAGED ? reinterpret_cast<const int*>(slots)[2 * at] : at;
        };
#pragma unroll
        for (int p = 0; p < PIECES; ++p) krow[p] = row(kkey0[p]);
        vrow = row(vkey0);
    };
    auto set_tile = [&](int buf) {
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            const int kr = PAGED ? cache_row(krow[p], rows) : krow[p];
            const int vr = PAGED ? cache_row(vrow, rows) : vrow;
            ksrc[p] = kbase + (size_t)kr * ks * 2 + k_byte[p];
            vsrc[p] = vbase + (size_t)vr * vs * 2 + v_byte[p];
            m0k_cur[p] = m0k[buf][p];
            m0v_cur[p] = m0v[buf][p];
        }
    };
    auto stage = [&]() {
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            lds_transfer16(m0k_cur[p], ksrc[p]);
            lds_transfer16(m0v_cur[p], vsrc[p]);
        }
    };
    auto drain = [&]() {
        static_assert(PIECES == 4, "drain operand list");
        asm volatile("s_waitcnt vmcnt(0)"
                     :
                     : "v"(ksrc[0]), "v"(ksrc[1]), "v"(ksrc[2]), "v"(ksrc[3]),
                       "v"(vsrc[0]), "v"(vsrc[1]), "v"(vsrc[2]), "v"(vsrc[3]),
                       "s"(m0k_cur[0]), "s"(m0k_cur[1]), "s"(m0k_cur[2]),
                       "s"(m0k_cur[3]), "s"(m0v_cur[0]), "s"(m0v_cur[1]),
                       "s"(m0v_cur[2]), "s"(m0v_cur[3])
                     : "memory");
    };

    const int qpos = offset + qrow;                    // per-lane diagonal
    const int wave_kv_last = offset + qrow0 + QROWS;   // first key PAST the
                                                       // wave's last diagonal

    auto compute = [&](int t, const char* kbuf, const char* vbuf,
                       bool need_mask) {
        const int kv0 = t * KB;

        // ---- S^T = K·Q^T: 32x32 blocks of 32 keys ---------------------
        f32x16_t sa[NKB32];
        const f32x16_t zero = (f32x16_t)(0.0f);
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int kb = 0; kb < NKB32; ++kb) {
                uint4 ak = *reinterpret_cast<const uint4*>(
                    kbuf + k_swz_read(kb * 32 + l31, s * 32 + lh * 16));
                sa[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    *reinterpret_cast<bf16x8_t*>(&ak),
                    *reinterpret_cast<bf16x8_t*>(&bq[s]), s ? sa[kb] : zero, 0, 0, 0);
            }

        // ---- mask + online softmax (per-lane row, RAW-score domain) --------
        // lane's score i of block kb = key kv0 + kb*32 + (i&3) + 8*(i>>2) + 4*lh
        // Scores stay UNSCALED: scale*log2(e) folds into the exp2 argument
        // (one v_fma per score instead of a separate scale pass + expf's
        // internal log2e multiply — v_exp_f32 IS exp2).
        const float scale2 = scale * 1.4426950408889634f;
        if (need_mask) {  // wave-uniform: one branch, not per-score selects.
            // Fold the tile-varying part into two per-lane values so each
            // score masks with compares against inline constants (keeping
            // the 64 kg values out of SGPRs — they spilled as writelanes).
            const int dqk = 4 * lh + kv0 - qpos;   // mask if dqk + c > 0
            const int dskv = 4 * lh + kv0 - Skv;   // mask if dskv + c >= 0
#pragma unroll
            for (int kb = 0; kb < NKB32; ++kb)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int c = kb * 32 + (i & 3) + 8 * (i >> 2);
                    if (dqk > -c || dskv >= -c) sa[kb][i] = -INFINITY;
                }
        }
        float rowmax = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < NKB32; ++kb)
#pragma unroll
            for (int i = 0; i < 16; ++i) rowmax = fmaxf(rowmax, sa[kb][i]);
        // half-wave exchange on the VALU (v_permlane32_swap), not ds_bpermute:
        // the LDS pipe stays free for the b128/tr16 operand reads
        rowmax = fmaxf(rowmax, xor32_f32(rowmax, lh));

        const float m_old = m;
        const float mn = fmaxf(m_old, rowmax);
        m = mn;
        // a split may show a row none of its keys
        const float mnb = (SPLIT || KG > 1) && mn == -INFINITY ? 0.0f : mn * scale2;
        float psum = 0.0f;

        // ---- exp + pack to bf16 quads: pk[kb][g] = keys kb*32+g*8+4*lh+{0..3}
        uint32_t pk[NKB32][4][2];
#pragma unroll
        for (int kb = 0; kb < NKB32; ++kb)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float p0 = __builtin_amdgcn_exp2f(
                    __builtin_fmaf(sa[kb][g * 4 + 0], scale2, -mnb));
                float p1 = __builtin_amdgcn_exp2f(
                    __builtin_fmaf(sa[kb][g * 4 + 1], scale2, -mnb));
                float p2 = __builtin_amdgcn_exp2f(
                    __builtin_fmaf(sa[kb][g * 4 + 2], scale2, -mnb));
                float p3 = __builtin_amdgcn_exp2f(
                    __builtin_fmaf(sa[kb][g * 4 + 3], scale2, -mnb));
                psum += (p0 + p1) + (p2 + p3);
                asm("v_cvt_pk_bf16_f32 %0, %1, %2"
                    : "=v"(pk[kb][g][0]) : "v"(p0), "v"(p1));
                asm("v_cvt_pk_bf16_f32 %0, %1, %2"
                    : "=v"(pk[kb][g][1]) : "v"(p2), "v"(p3));
            }
        psum += xor32_f32(psum, lh);
        // rescale only when some lane's running max moved (wave vote): after
        // the first few tiles most tiles leave every row max unchanged and
        // the 64 accumulator multiplies + lsum scale are skipped outright
        if (__any(rowmax > m_old)) {
            const float alpha = (SPLIT || KG > 1) && mn == -INFINITY
                                    ? 1.0f : __builtin_amdgcn_exp2f((m_old - mn) * scale2);
            lsum *= alpha;
#pragma unroll
            for (int db = 0; db < 4; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i) oa[db][i] *= alpha;
        }
        lsum += psum;

        // ---- P·V: O^T[dim][q-row] via mfma(A=V^T, B=P^T) -------------------
        // k-step ks2 covers keys ks2*16 + lh*8 + {0..7}: the lower half's lanes have their own
        // quad e2 and the partner's, the upper half's the partner's quad e2 + 1 and their own,
        // which is what one swap of the quads' halves leaves in its two registers.
#pragma unroll
        for (int ks2 = 0; ks2 < KB / 16; ++ks2) {
            const int kb = ks2 >> 1, e2 = (ks2 & 1) * 2;
            const auto w0 = __builtin_amdgcn_permlane32_swap(pk[kb][e2][0], pk[kb][e2 + 1][0], false, false);
            const auto w1 = __builtin_amdgcn_permlane32_swap(pk[kb][e2][1], pk[kb][e2 + 1][1], false, false);
            union {
                uint32_t u[4];
                bf16x8_t v8;
            } pf;
            pf.u[0] = w0[0];
            pf.u[1] = w1[0];
            pf.u[2] = w0[1];
            pf.u[3] = w1[1];

            // V^T A-fragment: subtile tr16 reads — group-uniform 128-B runs
            // (fs_eff = (ks2&1)*2 + lh selects the key octet, col = l31&15)
            const int sub_row = ((ks2 & 1) * 2 + lh) * 16 + (l31 & 15);
#pragma unroll
            for (int db = 0; db < 4; ++db) {
                const char* sub =
                    vbuf + ((kb * 8) + db * 2 + (l31 >> 4)) * 1024;
                bf16x4v r0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
                    (__attribute__((address_space(3))) bf16x4v*)(sub +
                                                                 sub_row * 8));
                bf16x4v r1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
                    (__attribute__((address_space(3))) bf16x4v*)(sub + 512 +
                                                                 sub_row * 8));
                union {
                    struct { bf16x4v lo, hi; } p;
                    bf16x8_t v8;
                } bv;
                bv.p.lo = r0;
                bv.p.hi = r1;
                oa[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    bv.v8, pf.v8, oa[db], 0, 0, 0);
            }
        }
    };

    const int first = tile0 + gid;
    if (first < ntiles) {
        find_rows(first);
        set_tile(0);
        stage();
        if (PAGED) find_rows(first + KG);
    }
    const bool far = PAGED && ntiles - tile0 > 3 * KG;
    uint32_t touched[TOUCHES];
    if (far) {
        const int part = SPLIT ? CEIL_DIV(Skv, (int)gridDim.z) : Skv, key0 = SPLIT ? (int)blockIdx.z * part : 0;
        touch_rows(touched, kbase, vbase, slots, rows, (int64_t)ks * 2, (int64_t)vs * 2, min(key0, Skv - 1),
                   min(key0 + part, Skv), turn * groups + place / pairs, CEIL_DIV(Sq, QTILE_H) * groups);
    }
    // static priority for the second half of the waves: the younger 4 lose VALU
    // arbitration on every segment otherwise. The readfirstlane keeps the condition
    // provably wave-uniform (exec-masking is ignored by s_setprio).
    if (__builtin_amdgcn_readfirstlane(threadIdx.x) >= 256)
        __builtin_amdgcn_s_setprio(1);
    drain();
    if (far) asm volatile("" : : "v"(touched[0]), "v"(touched[1]), "v"(touched[2]), "v"(touched[3]));
    __syncthreads();
    // every group takes as many steps as the first, which may have one tile more
    int cur = 0;
    for (int t = first; t - gid < ntiles; t += KG, cur ^= 1) {
        const int kv0 = t * KB;
        if (t + KG < ntiles) {
            if (!PAGED) find_rows(t + KG);
            set_tile(cur ^ 1);
            stage();
            if (PAGED) find_rows(t + 2 * KG);
        }
        if (t < ntiles && kv0 < wave_kv_last) {  // wave-uniform: skip past-diagonal tiles
            // fully-unmasked tile: every key <= every lane's diagonal
            const bool need_mask =
                !(kv0 + KB <= offset + qrow0 + 1 && kv0 + KB <= Skv);
            compute(t, smem + cur * KBYTES, smem + voff + cur * KBYTES,
                    need_mask);
        }
        drain();
        __syncthreads();
    }

    // ---- key groups added up: each keeps 128 / KG channels and takes the other groups' sums
    // of them, behind the loop's last barrier. A wave's area is [64][lane]: its sums by
    // channel, and where its own would be its maximum and weight sum
    constexpr int NDB = 4 / KG;
    if constexpr (KG > 1) {
        float* const area = reinterpret_cast<float*>(lds) + wid * WAVE * 64 + lane;
        float* const mine = area + gid * NG * WAVE * 64;
        mine[gid * NDB * 16 * WAVE] = m;
        mine[(gid * NDB * 16 + 1) * WAVE] = lsum;
#pragma unroll
        for (int db = 0; db < 4; ++db) {
            if (db / NDB == gid) {
#pragma unroll
                for (int i = 0; i < 16; ++i) oa[db % NDB][i] = oa[db][i];
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) mine[(db * 16 + i) * WAVE] = oa[db][i];
            }
        }
        __syncthreads();
        const float scale2 = scale * 1.4426950408889634f;
        float mo[KG - 1], lo[KG - 1], both = m;
#pragma unroll
        for (int o = 0; o < KG - 1; ++o) {
            const int g = o + (o >= gid);
            mo[o] = area[(g * NG * 64 + g * NDB * 16) * WAVE];
            lo[o] = area[(g * NG * 64 + g * NDB * 16 + 1) * WAVE];
            both = fmaxf(both, mo[o]);
        }
        // a split that shows a row no key leaves zeros; elsewhere the softmax of nothing is NaN
        const bool none = both == -INFINITY && (SPLIT || ntiles <= tile0);
        const float a = none ? 1.0f : __builtin_amdgcn_exp2f((m - both) * scale2);
        m = both;
        lsum *= a;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) oa[db][i] *= a;
#pragma unroll
        for (int o = 0; o < KG - 1; ++o) {
            const int g = o + (o >= gid);
            const float c = none ? 1.0f : __builtin_amdgcn_exp2f((mo[o] - both) * scale2);
            lsum += lo[o] * c;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    oa[db][i] = __builtin_fmaf(
                        area[(g * NG * 64 + (gid * NDB + db) * 16 + i) * WAVE], c, oa[db][i]);
        }
    }
    const int dim0 = KG > 1 ? gid * 32 * NDB : 0;  // of the channels left in oa[0 .. NDB)

    if (SPLIT) {
        if (qrow < Sq) {
            const size_t row = ((size_t)blockIdx.z * B * Sq + (size_t)b * Sq + qrow) * Hq + h;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *reinterpret_cast<float4*>(po + row * DHEAD + dim0 + db * 32 + g * 8 + 4 * lh) =
                        make_float4(oa[db][g * 4], oa[db][g * 4 + 1], oa[db][g * 4 + 2], oa[db][g * 4 + 3]);
            if (lh == 0 && gid == 0) *reinterpret_cast<float2*>(pml + row * 2) = make_float2(m, lsum);
        }
        return;
    }
    // ---- epilogue: out[q-row][d] = o/l; lane holds dims (i&3)+8*(i>>2)+4*lh
    if (qrow < Sq) {
        const float inv_l = (lsum > 0.0f) ? 1.0f / lsum : 0.0f;
        uint16_t* op = out + ((size_t)(b * Sq + qrow) * Hq + h) * DHEAD;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int d0 = dim0 + db * 32 + g * 8 + 4 * lh;
                uint2 pkd;
                pkd.x = (uint32_t)f32_to_bf16(oa[db][g * 4 + 0] * inv_l) |
                        ((uint32_t)f32_to_bf16(oa[db][g * 4 + 1] * inv_l) << 16);
                pkd.y = (uint32_t)f32_to_bf16(oa[db][g * 4 + 2] * inv_l) |
                        ((uint32_t)f32_to_bf16(oa[db][g * 4 + 3] * inv_l) << 16);
                *reinterpret_cast<uint2*>(op + d0) = pkd;
            }
    }
}

// The sums of a row in one order of the keys, 128 queries of a head a block: for callers that
// quantise what follows. There another rounding of a weight moves activations to the
// next 8-bit value, and two forms that are each 0.036 from 64 bits end 0.037 apart; so 8-bit
// models keep the form and the splits that they had, whatever is the fastest. Waves of
// 16 rows on 16x16x32 products; P goes through LDS to become an operand. A tile takes 5 us,
// its LDS reads (512 KB for 128 rows) the most of it. It alone takes its maxima of scaled scores, which
// scales of 0 and below need.
template <bool SPLIT, bool PAGED>
__global__ __launch_bounds__(512, 1) void attn_prefill_steady_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
    const uint16_t* __restrict__ v, uint16_t* __restrict__ out, int B, int Hq,
    int Hk, int Sq, int Skv, float scale, int qs, int ks, int vs,
    float* __restrict__ po, float* __restrict__ pml, const int64_t* __restrict__ slots, int rows) {
    constexpr int KB = 128, QROWS = 16;
    constexpr int QTILE = QROWS * NWAVE;
    constexpr int P_BYTES = QROWS * KB * 2;
    constexpr int KBYTES = KB * DHEAD * 2;   // one K (or V) ring buffer
    constexpr int PIECES = KB / 32;          // 1-KiB DMA chunks per wave
    constexpr int NKB = KB / 16;             // 16-key QK column blocks
    constexpr int NKB2 = KB / 32;            // 32-key PV k-blocks
    __shared__ __attribute__((aligned(16))) char smem[4 * KBYTES +
                                                      NWAVE * P_BYTES];
    const uint32_t voff = 2 * KBYTES;        // V buffers after the K ring
    const uint32_t poff = voff + 2 * KBYTES;

    const int groups = Hq / Hk, pairs = B * Hk, nbh = pairs * groups;
    const int turn = blockIdx.x / nbh, place = blockIdx.x % nbh;
    const int qtile = CEIL_DIV(Sq, QTILE) - 1 - turn;        // as in attn_prefill_kernel
    const int bh = place % pairs * groups + place / pairs;
    const int b = bh / Hq;
    const int h = bh % Hq;
    const int hk = h / (Hq / Hk);
    const int offset = Skv - Sq;  // causal diagonal offset

    const int tid = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int wid = tid / WAVE;
    const int fr = lane & 15;  // fragment row/col index (0..15)
    const int fs = lane >> 4;  // k-slice 0..3

    // ---- Q fragments: aq[dblk] = Q[qrow0 + fr][d = dblk*32 + fs*8]
    const int qrow0 = qtile * QTILE + wid * QROWS;
    uint4 aq[4];
    if (qrow0 + fr < Sq) {
        const uint16_t* qp = q + (size_t)(b * Sq + qrow0 + fr) * qs + (size_t)h * DHEAD;
#pragma unroll
        for (int dblk = 0; dblk < 4; ++dblk)
            aq[dblk] = *reinterpret_cast<const uint4*>(qp + dblk * 32 + fs * 8);
    } else {
#pragma unroll
        for (int dblk = 0; dblk < 4; ++dblk) aq[dblk] = make_uint4(0, 0, 0, 0);
    }

    float m[4], lsum[4];
    f32x4_t o_acc[8];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        m[r] = -INFINITY;
        lsum[r] = 0.0f;
    }
#pragma unroll
    for (int nb = 0; nb < 8; ++nb) o_acc[nb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

    const int kv_needed = min(Skv, offset + qtile * QTILE + QTILE);
    const int all_tiles = CEIL_DIV(max(kv_needed, 0), KB);
    const int run = SPLIT ? CEIL_DIV(all_tiles, (int)gridDim.z) : all_tiles;
    const int tile0 = SPLIT ? (int)blockIdx.z * run : 0;
    const int ntiles = SPLIT ? min(all_tiles, tile0 + run) : all_tiles;

    const char* kbase = reinterpret_cast<const char*>(k) +
                        ((size_t)b * Skv * ks + (size_t)hk * DHEAD) * 2;
    const char* vbase = reinterpret_cast<const char*>(v) +
                        ((size_t)b * Skv * vs + (size_t)hk * DHEAD) * 2;

    const int skv_clamp = Skv - 1;

    // transfers as in attn_prefill_kernel
    // per-piece invariants
    // a wave's pieces of V are channels of the same keys
    int k_byte[PIECES], v_byte[PIECES], kkey0[PIECES], vkey0 = 0;
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
        const int c = wid * PIECES + p;
        const int kkey = c * 4 + (lane >> 4);
        kkey0[p] = kkey;
        k_byte[p] = ((lane & 15) * 16) ^ ((kkey & 15) << 4);
        const int kb2 = c >> 3, nb = c & 7;
        vkey0 = kb2 * 32 + v_img_row_inv(lane >> 1);
        v_byte[p] = (nb * 16 + (lane & 1) * 8) * 2;
    }
    // LDS destinations (uniform per wave): [buf][piece] for K and V
    uint32_t m0k[2][PIECES], m0v[2][PIECES];
#pragma unroll
    for (int buf = 0; buf < 2; ++buf)
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            const int c = wid * PIECES + p;
            m0k[buf][p] = __builtin_amdgcn_readfirstlane(
                (uint32_t)(uintptr_t)smem + buf * KBYTES + c * 1024);
            m0v[buf][p] = __builtin_amdgcn_readfirstlane(
                (uint32_t)(uintptr_t)smem + voff + buf * KBYTES + c * 1024);
        }
    // persistent asm operands: current tile's source addresses + LDS bases
    const char* ksrc[PIECES];
    const char* vsrc[PIECES];
    uint32_t m0k_cur[PIECES], m0v_cur[PIECES];
    // PAGED: the rows of a tile are looked up a tile ahead of its transfers, straight-line and
    // as loaded, so that the only wait for them is the drain
    int krow[PIECES], vrow = 0;
    auto find_rows = [&](int t) {
        const int kv0 = t * KB;
        auto row = [&](int key) {
            const int at = min(kv0 + key, skv_clamp);
            return PAGED ? reinterpret_cast<const int*>(slots)[2 * at] : at;
        };
#pragma unroll
        for (int p = 0; p < PIECES; ++p) krow[p] = row(kkey0[p]);
        vrow = row(vkey0);
    };
    auto set_tile = [&](int buf) {
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            const int kr = PAGED ? cache_row(krow[p], rows) : krow[p];
            const int vr = PAGED ? cache_row(vrow, rows) : vrow;
            ksrc[p] = kbase + (size_t)kr * ks * 2 + k_byte[p];
            vsrc[p] = vbase + (size_t)vr * vs * 2 + v_byte[p];
            m0k_cur[p] = m0k[buf][p];
            m0v_cur[p] = m0v[buf][p];
        }
    };
    auto stage = [&]() {
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            lds_transfer16(m0k_cur[p], ksrc[p]);
            lds_transfer16(m0v_cur[p], vsrc[p]);
        }
    };

    auto compute = [&](int t, const char* kbuf, const char* vbuf) {
        const int kv0 = t * KB;
        const bool need_mask = !(kv0 + KB <= offset + qrow0 + 1 && kv0 + KB <= Skv);

        // ---- QK^T ----------------------------------------------------
        f32x4_t s[NKB];
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
            f32x4_t acc = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int dblk = 0; dblk < 4; ++dblk) {
                uint4 bk = *reinterpret_cast<const uint4*>(
                    kbuf + k_swz_read(kb * 16 + fr, (dblk * 32 + fs * 8) * 2));
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    *reinterpret_cast<bf16x8_t*>(&aq[dblk]),
                    *reinterpret_cast<bf16x8_t*>(&bk), acc, 0, 0, 0);
            }
            s[kb] = acc;
        }

        // ---- mask + online softmax -----------------------------------
        const int qpos = offset + qrow0 + fs * 4;  // + reg
        float rowmax[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) rowmax[r] = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
#pragma unroll
            for (int r = 0; r < 4; ++r) s[kb][r] *= scale;
        }
        if (need_mask) {  // wave-uniform
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb) {
                const int kg = kv0 + kb * 16 + fr;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (kg > qpos + r || kg >= Skv) s[kb][r] = -INFINITY;
            }
        }
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
#pragma unroll
            for (int r = 0; r < 4; ++r) rowmax[r] = fmaxf(rowmax[r], s[kb][r]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) rowmax[r] = group16_reduce_max(rowmax[r]);

        float alpha[4], psum[4], mref[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float mn = fmaxf(m[r], rowmax[r]);
            // a split may show a row none of its keys
            mref[r] = SPLIT && mn == -INFINITY ? 0.0f : mn;
            alpha[r] = __expf(m[r] - mref[r]);
            m[r] = mn;
            psum[r] = 0.0f;
        }
        // fully-masked padding rows produce NaN locally, never stored.

#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float p = __expf(s[kb][r] - mref[r]);
                s[kb][r] = p;
                psum[r] += p;
                *reinterpret_cast<uint16_t*>(
                    smem + poff + wid * P_BYTES +
                    (fs * 4 + r) * (KB * 2) +
                    (((kb * 16 + fr) * 2) ^ (((fs * 4 + r) & 7) << 4))) =
                    f32_to_bf16(p);
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            psum[r] = group16_reduce_sum(psum[r]);
            lsum[r] = lsum[r] * alpha[r] + psum[r];
        }
#pragma unroll
        for (int nb = 0; nb < 8; ++nb)
#pragma unroll
            for (int r = 0; r < 4; ++r) o_acc[nb][r] *= alpha[r];

        // ---- P·V (V via hardware transpose reads) --------------------
        uint4 ap[NKB2];
#pragma unroll
        for (int kb2 = 0; kb2 < NKB2; ++kb2) {
            const int prow = fr;
            ap[kb2] = *reinterpret_cast<const uint4*>(
                smem + poff + wid * P_BYTES + prow * (KB * 2) +
                (((kb2 * 32 + fs * 8) * 2) ^ ((prow & 7) << 4)));
        }
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) {
#pragma unroll
            for (int kb2 = 0; kb2 < NKB2; ++kb2) {
                bf16x4v r0, r1;
                const char* sub = vbuf + (kb2 * 8 + nb) * 1024;
                r0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
                    (__attribute__((address_space(3))) bf16x4v*)(sub + lane * 8));
                r1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
                    (__attribute__((address_space(3))) bf16x4v*)(sub + 512 + lane * 8));
                union {
                    struct { bf16x4v lo, hi; } p;
                    bf16x8_t v8;
                } bv;
                bv.p.lo = r0;
                bv.p.hi = r1;
                o_acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    *reinterpret_cast<bf16x8_t*>(&ap[kb2]), bv.v8,
                    o_acc[nb], 0, 0, 0);
            }
        }
    };

    auto drain = [&]() {
        static_assert(PIECES == 4, "drain operand list");
        asm volatile("s_waitcnt vmcnt(0)"
                     :
                     : "v"(ksrc[0]), "v"(ksrc[1]), "v"(ksrc[2]), "v"(ksrc[3]),
                       "v"(vsrc[0]), "v"(vsrc[1]), "v"(vsrc[2]), "v"(vsrc[3]),
                       "s"(m0k_cur[0]), "s"(m0k_cur[1]), "s"(m0k_cur[2]),
                       "s"(m0k_cur[3]), "s"(m0v_cur[0]), "s"(m0v_cur[1]),
                       "s"(m0v_cur[2]), "s"(m0v_cur[3])
                     : "memory");
    };
    if (ntiles > tile0) {
        find_rows(tile0);
        set_tile(0);
        stage();
        if (PAGED) find_rows(tile0 + 1);
    }
    const bool far = PAGED && ntiles - tile0 > 3;
    uint32_t touched[TOUCHES];
    if (far) {
        const int part = SPLIT ? CEIL_DIV(Skv, (int)gridDim.z) : Skv, key0 = SPLIT ? (int)blockIdx.z * part : 0;
        touch_rows(touched, kbase, vbase, slots, rows, (int64_t)ks * 2, (int64_t)vs * 2, min(key0, Skv - 1),
                   min(key0 + part, Skv), turn * groups + place / pairs, CEIL_DIV(Sq, QTILE) * groups);
    }
    if (__builtin_amdgcn_readfirstlane(threadIdx.x) >= 256)
        __builtin_amdgcn_s_setprio(1);
    drain();
    if (far) asm volatile("" : : "v"(touched[0]), "v"(touched[1]), "v"(touched[2]), "v"(touched[3]));
    __syncthreads();
    for (int t = tile0; t < ntiles; ++t) {
        const int cur = (t - tile0) & 1;
        if (t + 1 < ntiles) {
            if (!PAGED) find_rows(t + 1);
            set_tile(cur ^ 1);
            stage();
            if (PAGED) find_rows(t + 2);
        }
        compute(t, smem + cur * KBYTES, smem + voff + cur * KBYTES);
        drain();          // tile t+1 has landed
        __syncthreads();  // all waves' reads of buf[cur] complete
    }

    // ---- epilogue: out[row][d] = o / l ------------------------------------
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = qrow0 + fs * 4 + r;
        if (row >= Sq) continue;
        if (SPLIT) {
            const size_t at = ((size_t)blockIdx.z * B * Sq + (size_t)b * Sq + row) * Hq + h;
#pragma unroll
            for (int nb = 0; nb < 8; ++nb) po[at * DHEAD + nb * 16 + fr] = o_acc[nb][r];
            if (fr == 0) *reinterpret_cast<float2*>(pml + at * 2) = make_float2(m[r], lsum[r]);
            continue;
        }
        const float inv_l = (lsum[r] > 0.0f) ? 1.0f / lsum[r] : 0.0f;
        uint16_t* op = out + ((size_t)(b * Sq + row) * Hq + h) * DHEAD;
#pragma unroll
        for (int nb = 0; nb < 8; ++nb)
            op[nb * 16 + fr] = f32_to_bf16(o_acc[nb][r] * inv_l);
    }
}

// Splits added up: one wave per (query, head) row, two channels per lane. rows = B * Sq
// * Hq; scale2 turns a difference of maxima (of unscaled scores but in the steady form) into a
// power of two. A split without a visible
// key has weight sum 0; one with a NaN or an infinite score has a NaN sum, and counts.
// The launch is its chain of loads: the first eight splits are asked for together, weights
// or not (77 queries of 32 heads behind 1187 keys, 8 splits: 7.4 us -> 3.9).
__global__ __launch_bounds__(256) void prefill_combine_kernel(const float* __restrict__ po,
                                                              const float* __restrict__ pml,
                                                              uint32_t* __restrict__ out, int rows,
                                                              int nsplit, float scale2) {
    const int row = blockIdx.x * 4 + threadIdx.x / WAVE, lane = threadIdx.x & (WAVE - 1);
    if (row >= rows) return;
    constexpr int AHEAD = 8;
    auto stats = [&](int s) {
        return *reinterpret_cast<const float2*>(pml + ((size_t)s * rows + row) * 2);
    };
    auto part = [&](int s) {
        return *reinterpret_cast<const float2*>(po + ((size_t)s * rows + row) * DHEAD + lane * 2);
    };
    float2 ml[AHEAD], o[AHEAD];
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) {
        ml[s] = stats(min(s, nsplit - 1));
        o[s] = part(min(s, nsplit - 1));
    }
    float mx = -INFINITY;
#pragma unroll
    for (int s = 0; s < AHEAD; ++s)
        if (s < nsplit && ml[s].y != 0.0f) mx = fmaxf(mx, ml[s].x);
    for (int s = AHEAD; s < nsplit; ++s) {
        const float2 m = stats(s);
        if (m.y != 0.0f) mx = fmaxf(mx, m.x);
    }
    float l = 0.0f, a = 0.0f, b = 0.0f;
    auto add = [&](const float2& m, const float2& v) {
        const float w = __builtin_amdgcn_exp2f((m.x - mx) * scale2);
        l = fmaf(m.y, w, l);
        a = fmaf(v.x, w, a);
        b = fmaf(v.y, w, b);
    };
#pragma unroll
    for (int s = 0; s < AHEAD; ++s)
        if (s < nsplit && ml[s].y != 0.0f) add(ml[s], o[s]);
    for (int s = AHEAD; s < nsplit; ++s) {
        const float2 m = stats(s);
        if (m.y != 0.0f) add(m, part(s));
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    out[(size_t)row * (DHEAD / 2) + lane] = pack_bf16x2(a * inv, b * inv);
}

// Key-split forms: merged = 0, a block per head and 128 queries (64 up to 64 queries); 1, a
// block per key head and 256 / (Hq / Hk) queries (Hq / Hk of 2, 4 or 8); 2, the steady form.
// po [nsplit, B, Sq, Hq, 128] and pml [nsplit, B, Sq, Hq, 2]: float32 scratch.
#define LAUNCH_PREFILL(KG, GQ, SPLIT, NSPLIT)                                                      \
    do {                                                                                           \
        if (slots) LAUNCH_BLOCKS((attn_prefill_kernel<KG, GQ, SPLIT, true>), 256 / (KG) / (GQ), B * (Hq / (GQ)), NSPLIT); \
        else LAUNCH_BLOCKS((attn_prefill_kernel<KG, GQ, SPLIT, false>), 256 / (KG) / (GQ), B * (Hq / (GQ)), NSPLIT); \
    } while (0)
#define LAUNCH_STEADY(SPLIT, NSPLIT)                                                               \
    do {                                                                                           \
        if (slots) LAUNCH_BLOCKS((attn_prefill_steady_kernel<SPLIT, true>), 128, B * Hq, NSPLIT);  \
        else LAUNCH_BLOCKS((attn_prefill_steady_kernel<SPLIT, false>), 128, B * Hq, NSPLIT);       \
    } while (0)
#define LAUNCH_BLOCKS(KERN, ROWS, HEADS, NSPLIT)                                                   \
    hipLaunchKernelGGL(KERN, dim3(CEIL_DIV(Sq, ROWS) * (HEADS), 1, NSPLIT),                        \
                       dim3(512), 0, (hipStream_t)stream, (const uint16_t*)q, (const uint16_t*)k,  \
                       (const uint16_t*)v, (uint16_t*)out, B, Hq, Hk, Sq, Skv, scale, q_stride,    \
                       k_stride, v_stride, (float*)po, (float*)pml, (const int64_t*)slots, cache_rows)

extern "C" int oa_attention_prefill_split(
    void* stream, const void* q, const void* k, const void* v, void* out, void* po, void* pml,
    int B, int Hq, int Hk, int Sq, int Skv, int D, float scale, int q_stride, int k_stride,
    int v_stride, int nsplit, int merged, const void* slots, int cache_rows) {
    if (D != DHEAD) return -100;
    if (Hk < 1 || Hq % Hk != 0) return -101;
    if ((q_stride | k_stride | v_stride) % 8 != 0) return -102;
    if (slots && (B != 1 || cache_rows < 1)) return -106;
    if (nsplit < 1 || nsplit > 65535 || (int64_t)B * Sq * Hq > (1 << 30)) return -105;
    const int gq = Hq / Hk, rows = B * Sq * Hq;
    if (rows < 1) return 0;
    if (merged == 2) {
        LAUNCH_STEADY(true, nsplit);
    }
    else if (!merged) {
        if (Sq <= 64) LAUNCH_PREFILL(4, 1, true, nsplit);
        else LAUNCH_PREFILL(2, 1, true, nsplit);
    }
    else if (gq == 2) LAUNCH_PREFILL(1, 2, true, nsplit);
    else if (gq == 4) LAUNCH_PREFILL(1, 4, true, nsplit);
    else if (gq == 8) LAUNCH_PREFILL(1, 8, true, nsplit);
    else return -104;
    HIP_CHECK_LAUNCH();
    hipLaunchKernelGGL(prefill_combine_kernel, dim3(CEIL_DIV(rows, 4)), dim3(256), 0,
                       (hipStream_t)stream, (const float*)po, (const float*)pml, (uint32_t*)out, rows,
                       nsplit, merged == 2 ? 1.4426950408889634f : scale * 1.4426950408889634f);
    HIP_CHECK_LAUNCH();
    return 0;
}

extern "C" int oa_attention_prefill_variant(
    void* stream, const void* q, const void* k, const void* v, void* out,
    int B, int Hq, int Hk, int Sq, int Skv, int D, float scale,
    int q_stride, int k_stride, int v_stride, int variant, const void* slots, int cache_rows) {
    if (D != DHEAD) return -100;
    if (Hq % Hk != 0) return -101;
    if ((q_stride | k_stride | v_stride) % 8 != 0) return -102;
    if (slots && (B != 1 || cache_rows < 1)) return -106;
    float* const po = nullptr;
    float* const pml = nullptr;
    switch (variant) {
        case 7:  // the steady form, 128 rows
            LAUNCH_STEADY(false, 1);
            break;
        case 10:  // two key groups, 128 rows
            LAUNCH_PREFILL(2, 1, false, 1);
            break;
        case 11:  // four key groups, 64 rows
            LAUNCH_PREFILL(4, 1, false, 1);
            break;
        case 8:  // 256 rows of one head
            LAUNCH_PREFILL(1, 1, false, 1);
            break;
        case 9:  // 256 rows: the q-heads of a KV head share each staged KV tile
            if (Hq == 2 * Hk)
                LAUNCH_PREFILL(1, 2, false, 1);
            else if (Hq == 4 * Hk)
                LAUNCH_PREFILL(1, 4, false, 1);
            else if (Hq == 8 * Hk)
                LAUNCH_PREFILL(1, 8, false, 1);
            else
                return -104;
            break;
        default:
            return -103;
    }
    HIP_CHECK_LAUNCH();
    return 0;
}

// Time of KG key groups without key splits in us, over 256 CUs: a chain of 128-key tiles is the
// longest block's, or, where there are more blocks than CUs, the chip's share of all tiles
// and half a block for the uneven end. Over 170 sizes (1 to 64 heads, 16 to 4096 queries,
// up to 9000 keys) the form it names took 0.1 per cent more than the best of the three,
// 19 at the most (64 blocks of 282 queries: 16.4 for 13.8).
static float prefill_us(int kg, int B, int Hq, int Sq, int Skv) {
    const float tile = kg == 1 ? 4.2f : kg == 2 ? 2.6f : 2.0f;
    const int qt = 256 / kg, nq = CEIL_DIV(Sq, qt);
    const float last = CEIL_DIV(Skv, 128), blocks = (float)nq * B * Hq;
    const float first = nq > 1 ? fminf(CEIL_DIV(Skv - Sq + qt, 128), last) : last;
    const float mean = (first + last) / 2;
    return tile * (blocks <= 256 ? last : fmaxf(last, mean * (blocks / 256 + 0.5f)));
}

extern "C" int oa_attention_prefill(void* stream, const void* q, const void* k,
                                    const void* v, void* out, int B, int Hq,
                                    int Hk, int Sq, int Skv, int D, float scale,
                                    int q_stride, int k_stride, int v_stride, int steady,
                                    const void* slots, int cache_rows) {
    // OPSAGENT_PREFILL_VARIANT (7 to 11, 9 where heads are shared) forces a variant
    // (read per call so one process can A/B all variants).
    const char* e = getenv("OPSAGENT_PREFILL_VARIANT");
    int variant = e ? atoi(e) : 0;
    const int gq = (Hk > 0 && Hq % Hk == 0) ? Hq / Hk : 1;
    const bool shared = gq == 2 || gq == 4 || gq == 8;
    if (variant <= 0 && !(scale > 0.0f)) {
        variant = 7;     // the maximum of scores that are scaled; the others scale maxima
    } else if (variant <= 0 && steady) {
        const int64_t heads = (int64_t)B * Hq;
        variant = shared && CEIL_DIV(Sq, 128) * heads > 256 ? 9
                  : CEIL_DIV(Sq, 256) * heads >= 256 ? 8 : 7;
    } else if (variant <= 0) {
        const float one = prefill_us(1, B, Hq, Sq, Skv), two = prefill_us(2, B, Hq, Sq, Skv),
                    four = prefill_us(4, B, Hq, Sq, Skv);
        variant = four <= two && four <= one ? 11 : two <= one ? 10 : shared ? 9 : 8;
    }
    return oa_attention_prefill_variant(stream, q, k, v, out, B, Hq, Hk, Sq,
                                        Skv, D, scale, q_stride, k_stride,
                                        v_stride, variant, slots, cache_rows);
}
