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
// Launches of under 512 (sequence, key head) pairs: a split is `chunk` keys, a multiple of 64 (decode_chunk), and blocks past a
// sequence's last key end at once. Larger ones: the tiles of 64 keys of all sequences are cut in
// equal runs, one a CU (DecodeRuns). Either way at most nsplit splits cover a sequence, and the
// combine reads those that exist: plain splits it counts, behind a sequence's last run stands a mark.

#include <type_traits>

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

// halves (DIST 32) or neighbouring rows of 16 lanes (16) of a and b added up: the lanes of
// the first half (row) get a's sum, those of the second b's
template <int DIST>
__device__ __forceinline__ float swap_add(float a, float b) {
    const auto r = DIST == 32
        ? __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false)
        : __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// A batch is padded to the size of a captured step with copies of its first row. Such a
// row is told by its slot (no other two rows write one), and that it is one is then seen
// from all that its result depends on: length, pages and, for its key head, the bits of
// queries, key and value. It leaves a mark for the combine, which reads the first row's
// partial results in its place. Both launches, us: 47 rows of up to 3000 tokens in a step
// of 64 100.2 -> 88.9, 33 of up to 1500 54.3 -> 42.7, 24 of up to 2000 in 32 40.7 -> 38.8;
// a full step pays for the look: 64 of up to 3000 112.3 -> 112.8, of up to 300 22.1 -> 22.5.
// (With splits of each sequence; runs leave such rows out and look at them in blocks of their own.)
//
// Marks stand where a sum of weights would be: of a copy's first split, with runs of the place behind
// a row's last one.
#define COPY_MARK -1.0f
#define END_MARK -2.0f
template <int G>
__device__ __forceinline__ bool copy_of_first(const uint32_t* q, int qs2, const uint32_t* kin, int ks2,
                                              const uint32_t* vin, int vs2, const int* block_table,
                                              int max_blocks, int b, int h, int pages) {
    const int lane = threadIdx.x & (WAVE - 1);
    uint32_t diff = 0;
    for (int i = lane; i < G * DHEAD / 2; i += WAVE)
        diff |= q[(size_t)b * qs2 + h * G * DHEAD / 2 + i] ^ q[h * G * DHEAD / 2 + i];
    const int kv = h * DHEAD / 2 + lane;
    diff |= (kin[(size_t)b * ks2 + kv] ^ kin[kv]) | (vin[(size_t)b * vs2 + kv] ^ vin[kv]);
    for (int i = lane; i < pages; i += WAVE)
        diff |= block_table[(size_t)b * max_blocks + i] ^ block_table[i];
    return !__any(diff != 0);
}

// 16 bytes of a value row. NT: in a busy step it is read once, and all of it by one load: without
// being kept. 47 sequences of up to 3000 tokens 79.0 -> 74.5 us, 64 of 300 20.8 -> 20.6. The loads of
// key rows take a quarter of each at a time, from a line that has to stay meanwhile: with nt 5%
// slower. The rows of few sequences stay in the last cache from step to step: an agent's turn of an 8B
// model 59.1 -> 60.9 ms with nt.
template <bool NT>
__device__ __forceinline__ uint4 load_value(const uint32_t* p) {
    typedef __attribute__((ext_vector_type(4))) uint32_t u4;
    const u4* at = reinterpret_cast<const u4*>(p);
    return __builtin_bit_cast(uint4, NT ? __builtin_nontemporal_load(at) : *at);
}

// inclusive sums over the wave's lanes, by row shifts and row broadcasts
__device__ __forceinline__ int wave_sums(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
    return v;
}

// Whether row b may be a copy of the first one. (All loads at once: each wait for memory would
// add to every launch.)
__device__ __forceinline__ bool maybe_copy(const int* slots, const int* seq_lens, int b, int copies) {
    if (!copies) return false;
    const int n = seq_lens[b], n0 = seq_lens[0], slot = slots[b], slot0 = slots[0];
    return (b > 0) & (slot == slot0) & (n == n0);
}
// keys of row b in the runs
__device__ __forceinline__ int run_keys(const int* seq_lens, const int* slots, int b, int copies) {
    const int n = seq_lens[b];
    return maybe_copy(slots, seq_lens, b, copies) ? 0 : max(n, 0);
}
__device__ __forceinline__ int in_tiles(int keys) { return (keys + 63) >> 6; }

// Runs. Blocks that end at a sequence's end are unequal, and beyond one a CU they wait for memory
// that is busy anyway: what bounds a busy step's attention is the cache's rows (256 bytes each, pages
// in any order: loads alone run at 5.6 TB/s, 6.1 with value rows read without being kept), and
// prologues and uneven ends on top. So each of `runs` blocks of a key head takes `per` tiles of 64 keys, sequence after
// sequence; a row of t tiles lies in (t + per - 2) / per + 1 runs at the most, which `per` keeps to
// nsplit. Key heads go in step, head h on die h % 8.
//
// Each row that a run begins costs it a prologue and a merge. Where rows are short, a run is one
// unit of `size` tiles of a row instead (chunk_base keys, or as many as nsplit asks for; `per` is 1),
// in step: the rows' first units, then what is left of them. The line: tiles for each of runs and rows, 3.5, or 8
// where rows are more than the runs by a quarter. Both launches, us, caches that no cache holds, splits of each
// sequence / here, steps of 64, 4 heads a key head on 8: 47 of up to 3000 tokens 91.5 / 77.9, 33 of 1500 43.2 /
// 39.6, 64 of 3000 113 / 100; units: 64 of 300 22.7 / 21.1, of 700 36.8 / 35.7, 47 of 700 31.5 / 30.4, of 1000 39.4 / 39.4.
// What a launch works out first shows where neither gains: 40 of 700 30.2 / 31.0, 47 of 500 25.8 / 26.1, and in
// steps of 32 on 16 key heads 24 of 1000 with 256 in common 32.6 / 34.9. Runs for 384 or 768 blocks are slower (47
// of 3000 89, 89; 74.5 for 256), for 512 level (79.5), and so are two tiles ahead (79).
//
// Rows that share most of their pages (a prompt's common beginning) are read from the die's L2 by blocks that
// go in step, and runs would not: units, then, where the page at the mean length is the same. Splits of each
// sequence / runs / units, us: 64 of up to 1500 with 1024 in common 41.0 / 46.0 / 42.8, of 2200 with 2016 50.1 / 55.7 /
// 51.1, 56 of 1500 with 1024 39.6 / 42.6 / 39.5. With less in common runs stay ahead: 47 of 3000 with 256 83.3 / 72.1.
struct DecodeRuns {
    bool units;
    int size, per, total;
    int b, n;               // row (-1: none) and keys of it
    int before;             // tiles of the rows before it; units: `which` less the unit's number in its row
};

__device__ __forceinline__ int in_units(int t, int size) {
    return size & (size - 1) ? CEIL_DIV(t, size) : (t + size - 1) >> __builtin_ctz(size);
}

// The row that run `which` begins with. Every wave works it out for itself, a lane per sequence,
// 64 sequences at a time.
__device__ __forceinline__ DecodeRuns decode_runs(const int* seq_lens, const int* slots, const int* block_table,
                                                  int max_blocks, int block_shift, int B, int copies, int runs,
                                                  int nsplit, int chunk_base, int which, int whole) {
    const int lane = threadIdx.x & (WAVE - 1);
    auto keys = [&](int b) {
        const int n = run_keys(seq_lens, slots, min(b, B - 1), copies);
        return b < B ? n : 0;
    };
    DecodeRuns r;
    const int n0 = keys(lane);
    int most = n0, rows = __builtin_popcountll(__ballot(n0 > 0));
    r.total = __builtin_amdgcn_readlane(wave_sums(in_tiles(n0)), 63);
#pragma unroll 1
    for (int b0 = WAVE; b0 < B; b0 += WAVE) {
        const int n = keys(b0 + lane);
        most = max(most, n);
        rows += __builtin_popcountll(__ballot(n > 0));
        r.total += __builtin_amdgcn_readlane(wave_sums(in_tiles(n)), 63);
    }
    most = in_tiles(most);
    // (divisions only where they are needed: every launch waits for this)
    bool units = 2 * r.total < (4 * rows > 5 * runs ? 16 : 7) * (runs + rows);
    int cut = chunk_base / 64;
    if (!units) {
        // the page at the mean length: do half and more of the rows that are longer (of 64) have the same one?
        const int depth = (int)((float)(r.total * 64) * __builtin_amdgcn_rcpf((float)rows));
        const int page = block_table[(size_t)min(lane, B - 1) * max_blocks + min(depth >> block_shift, max_blocks - 1)];
        const uint64_t longer = __ballot(n0 > depth);
        const int first = __builtin_amdgcn_readlane(page, longer ? __builtin_ctzll(longer) : 0);
        const int same = __builtin_popcountll(longer & __ballot(page == first));
        units = same > 1 && 2 * same >= __builtin_popcountll(longer);
        const int fit = __builtin_amdgcn_readfirstlane(CEIL_DIV(r.total, units ? whole - B : runs));
        cut = units ? max(cut, fit) : fit;
    }
    const int over = units ? 0 : 1;
    while (const uint64_t more = __ballot(most - over > cut * (nsplit - over)))
        cut = CEIL_DIV(__builtin_amdgcn_readlane(most, __builtin_ctzll(more)) - over, nsplit - over);
    r.units = units;
    r.size = units ? cut : 1;
    r.per = units ? 1 : cut;
    r.b = -1;
    // units in step: the first ones of all rows, then, 64 rows at a time, the second ones and so on.
    // (Rows without keys have no place among them: blocks go to the CUs in turn, and such places would
    // leave some of them with less: 47 rows of up to 700 tokens in a step of 64 32.6 -> 30.3 us.)
    const bool firsts = units && which < rows;
    const int at = units ? which - (firsts ? 0 : rows) : which * r.per;
    int before = 0;
#pragma unroll 1
    for (int b0 = 0; b0 < B; b0 += WAVE) {
        const int n = b0 ? keys(b0 + lane) : n0, t = in_tiles(n);
        const int u = !units ? t : firsts ? min(t, 1) : max(in_units(t, r.size) - 1, 0);
        uint64_t some = __ballot(u > 0);
        const int sums = before + (firsts ? 0 : wave_sums(u));
        const int end = firsts ? before + __builtin_popcountll(some) : __builtin_amdgcn_readlane(sums, 63);
        if (end > at) {
            int unit = firsts ? 0 : 1, place = at - before;
            while (units && place >= __builtin_popcountll(some)) {
                place -= __builtin_popcountll(some);
                some = __ballot(u > unit++);
            }
            const uint64_t found = __ballot(units ? (some >> lane & 1) && __builtin_popcountll(some & ((1ull << lane) - 1)) == place
                                                  : sums > at);
            const int row = __builtin_ctzll(found);
            r.n = __builtin_amdgcn_readlane(n, row);
            r.b = b0 + row;
            r.before = units ? which - unit : __builtin_amdgcn_readlane(sums, row) - __builtin_amdgcn_readlane(u, row);
            break;
        }
        before = end;
    }
    return r;
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
// zeroed before every launch. copies: see copy_of_first. ROPE = true takes the raw projection outputs: the
// queries are rotated while they are split, the loop covers the CACHED keys
// [0, n-1), and the split that owns key n-1 rotates the new key, stores it and its
// value in the cache and starts its softmax with them. kin/vin/cs/sn/slots/kcw/vcw
// are only read when ROPE.
//
// PARTS (with ROPE, without runs): the projection is still its `splits` float32 planes [B, (Hq + 2 Hk) * 128],
// `plane` elements apart. A block adds up the columns of its heads, rounds them as the product alone
// would, and has them in LDS while its first keys and values are under way: what a launch for the sum took
// goes but for a barrier. us, that launch, this one and the combine / here: 8 sequences of up to 1500
// tokens, five planes 22.1 / 18.3 (traced one by one; a step of four layers 481.6 / 475.2).
struct Planes {
    const float* sums;
    int splits;
    int64_t plane;
};
struct Runs {
    int count;
};

// MORE: Runs with RUNS, otherwise Planes or nothing. (What a form has no use for is no argument: with a
// few bytes of such arguments here and in gemv1_kernel, decode steps of an 8B model took 2916 us, 2910 without.)
template <int G, bool FUSED, bool ROPE, bool RUNS, typename... MORE>
__global__ __launch_bounds__(256, RUNS && G <= 4 ? 3 : 1) void decode_attn_kernel(
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
    uint32_t* __restrict__ vcw, int ks2, int vs2, int copies, MORE... more) {
    constexpr bool PARTS = std::is_same_v<void(MORE...), void(Planes)>;
    static_assert(RUNS ? std::is_same_v<void(MORE...), void(Runs)> : PARTS || sizeof...(MORE) == 0, "one form");
    static_assert(!PARTS || (ROPE && !RUNS && !FUSED), "parts of a projection: plain launches only");
    constexpr int GP = G > 4 ? 8 : 4;            // columns of one part of the queries
    constexpr int KL = GP / 4;                   // keys per lane and tile
    // the (row, key head) in work and its keys; RUNS: tiles of the row, the first of them that
    // the block takes, and how many it still has to take
    int b, h, split, n, kstart, kend, own = 0, from = 0, left = 0;
    if constexpr (RUNS) {
        const int at = blockIdx.y, whole = gridDim.y - copies * (B - 1);
        h = blockIdx.x;
        split = 0;
        if (at < whole) {
            const DecodeRuns r = decode_runs(seq_lens, slots, block_table, max_blocks, block_shift, B, copies,
                                             more.count..., nsplit, chunk_base, at, whole);
            if (r.b < 0) return;
            b = r.b;
            n = r.n;
            own = in_tiles(n);
            if (r.units) {
                split = at - r.before;
                from = split * r.size;
                left = min(r.size, own - from);
            } else {
                from = at * r.per - r.before;
                left = min(r.per, r.total - at * r.per);
                split = __builtin_amdgcn_readfirstlane(at - r.before / r.per);
            }
        } else {                                     // a row that may be a copy, by itself if it is none
            b = 1 + at - whole;
            n = seq_lens[b];
            if (!maybe_copy(slots, seq_lens, b, copies) || n <= 0) return;
            left = own = in_tiles(n);
            if (copy_of_first<G>(q, qs2, kin, ks2, vin, vs2, block_table, max_blocks, b, h,
                                 (n + (1 << block_shift) - 1) >> block_shift)) {
                if (threadIdx.x < G) ml_part[((size_t)(b * Hk + h) * nsplit * G + threadIdx.x) * 2 + 1] = COPY_MARK;
                return;
            }
        }
    } else {
        b = blockIdx.x / Hk;
        h = blockIdx.x % Hk;
        split = blockIdx.y;
        n = seq_lens[b];
        const int chunk = decode_chunk(n, nsplit, chunk_base);
        kstart = split * chunk;
        if (!FUSED && kstart >= n) return;
        if (ROPE && copies && b > 0 && slots[b] == slots[0] && n == seq_lens[0] &&
            copy_of_first<G>(q, qs2, kin, ks2, vin, vs2, block_table, max_blocks, b, h,
                             CEIL_DIV(n, 1 << block_shift))) {
            if (split == 0 && threadIdx.x < G)
                ml_part[((size_t)blockIdx.x * nsplit * G + threadIdx.x) * 2 + 1] = COPY_MARK;
            return;
        }
        kend = min(n, kstart + chunk);
    }

    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int bmask = (1 << block_shift) - 1;
    __shared__ __attribute__((aligned(16))) float lds_o_[RUNS ? 2 : 1][4][G][DHEAD];
    __shared__ float lds_ml_[RUNS ? 2 : 1][4][G][2];

    // of a wave: its own range (of CACHED keys only; ROPE: the new key, index n - 1, is handled from
    // registers), whole tiles of 16
    int kend_c, wstart, wend, nt, page = 0;
    const int* btrow;
    auto range = [&]() {
        if (RUNS) {
            kstart = from * 64;
            kend = min(n, kstart + min(left, own - from) * 64);
        }
        kend_c = min(kend, ROPE ? n - 1 : n);
        const int span = max(kend_c - kstart, 0);
        const int wchunk = ((span + 63) >> 6) << 4;
        wstart = kstart + wid * wchunk;
        wend = min(kend_c, wstart + wchunk);
        nt = wend > wstart ? (wend - wstart + 15) >> 4 : 0;
        btrow = block_table + (size_t)b * max_blocks;
    };
    range();
    uint4 kr_[2][4], vr_[2][4];
#pragma unroll 1
    for (int row = 0;; ++row) {
    const int turn = row & 1;
    // (RUNS: what hangs on the lane alone is worked out for each row: kept, it costs a wave a SIMD)
    int lane = threadIdx.x & (WAVE - 1);
    if (RUNS) asm volatile("" : "+v"(lane));
    const int g16 = lane >> 4;   // row of 16 lanes: keys g16 * 4 .. + 3 of a tile
    const int dl = lane & 15;    // column; owns value channels dl*8 .. dl*8+7
    auto slot_of = [&](int kk) {
        return (int64_t)btrow[kk >> block_shift] << block_shift | (kk & bmask);
    };
    // A tile starts at a multiple of 16 keys: pages of 16 and more hold it whole, and
    // its page is one scalar load, made a tile ahead of the rows it leads to (47 sequences
    // of up to 3000 tokens, both launches: 93.2 us with five lookups per lane and tile
    // before its loads, 85.7; 8 of up to 1500 21.0, 20.1). Two tiles ahead cost a wave
    // per SIMD: 92.
    auto page_of = [&](int t) { return btrow[(wstart + min(t, nt - 1) * 16) >> block_shift]; };
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
        const uint32_t* vp[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) vp[i] = vc + ((size_t)vs[i] * Hk + h) * (DHEAD / 2) + dl * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) vw[i] = load_value<RUNS>(vp[i]);
    };
    // Loads return in order: the queries and their angles are asked for first, so that they
    // are rotated and split while the first keys, values and the new key are under way
    const int head = dl % GP, part = dl / GP;
    const bool have = head < G;
    __shared__ __attribute__((aligned(16))) uint32_t lds_in[PARTS ? (G + 2) * DHEAD / 2 : 4];
    constexpr int NIN = PARTS ? ((G + 2) * DHEAD / 4 + 255) / 256 : 1;    // four columns a thread and turn
    constexpr int NP = PARTS ? 8 : 1;            // planes asked for at once
    da_f4 in[NIN][NP];
    const da_f4* ip[NIN];
    if constexpr (PARTS) {
        const Planes planes(more...);
#pragma unroll
        for (int i = 0; i < NIN; ++i) {
            const int c = min((int)(i * 256 + threadIdx.x) * 4, (G + 2) * DHEAD - 4), at = c / DHEAD;
            const int col = (at < G ? h * G + at : Hk * G + (at - G) * Hk + h) * DHEAD + c % DHEAD;
            ip[i] = reinterpret_cast<const da_f4*>(planes.sums + (int64_t)b * (Hk * (G + 2) * DHEAD) + col);
#pragma unroll
            for (int k = 0; k < NP; ++k) in[i][k] = ip[i][min(k, planes.splits - 1) * (planes.plane / 4)];
        }
    }
    uint4 qw[4];
    if (!PARTS)
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
    auto load_first = [&]() {
        if (nt <= 0) return;
        load_tile(0, page_of(0), kr_[0], vr_[0]);
        page = page_of(1);
    };
    if (!RUNS || row == 0) load_first();
    if constexpr (PARTS) {
        const Planes planes(more...);
#pragma unroll
        for (int i = 0; i < NIN; ++i) {
            const int c = (i * 256 + threadIdx.x) * 4;
            da_f4 sum = in[i][0];
#pragma unroll
            for (int k = 1; k < NP; ++k)
                if (k < planes.splits) sum += in[i][k];
            for (int k = NP; k < planes.splits; ++k) sum += ip[i][k * (planes.plane / 4)];
            if (c < (G + 2) * DHEAD)
                *reinterpret_cast<uint2*>(&lds_in[c / 2]) =
                    make_uint2(pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3]));
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 4; ++s)
            qw[s] = *reinterpret_cast<const uint4*>(&lds_in[((have ? head : 0) * DHEAD + s * 32 + g16 * 8) / 2]);
    }
    const bool owner = ROPE && n - 1 >= kstart && n - 1 < kend && wid == 3;   // of the new key
    uint4 nk[4], nv;
    if (PARTS && owner) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
            nk[s] = *reinterpret_cast<const uint4*>(&lds_in[(G * DHEAD + s * 32 + g16 * 8) / 2]);
        nv = *reinterpret_cast<const uint4*>(&lds_in[((G + 1) * DHEAD + dl * 8) / 2]);
    } else if (owner) {
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

    const int bh = b * Hk + h;
    float* opart_row = o_part + ((size_t)(bh * nsplit + split) * G) * DHEAD;
    float* mlpart_row = ml_part + ((size_t)(bh * nsplit + split) * G) * 2;
    const bool last = RUNS && kend == n && split + 1 < nsplit;    // of a row's splits, and not of all places
    auto next = [&]() {
        left -= own - from;
        if (left <= 0) return;
        do n = run_keys(seq_lens, slots, ++b, copies);
        while (n == 0);
        own = in_tiles(n);
        from = split = 0;
        range();
        load_first();
    };
    if (RUNS) next();

    // sums and maxima of every head to all lanes of a row
    if (GP == 4) lsum += row_ror<4>(lsum);
    lsum += row_ror<8>(lsum);
    // Merge the wave's 4 rows: to their common maximum, then lane by lane. Swapping halves
    // (quarters) of two registers and adding them leaves each lane with half (a quarter) of
    // the sums, so that 24 swaps and as many additions do for G = 4 what took 80 exchanges
    // through the LDS
    float mt4 = fmaxf(m, __shfl_xor(m, 16, WAVE));
    mt4 = fmaxf(mt4, __shfl_xor(mt4, 32, WAVE));
    const float a4 = __expf(m - (mt4 == -INFINITY ? 0.0f : mt4));
    lsum *= a4;
    lsum += __shfl_xor(lsum, 16, WAVE);
    lsum += __shfl_xor(lsum, 32, WAVE);
    float al4[8];
    al4[0] = row_bcast<0>(a4); al4[1] = row_bcast<1>(a4);
    al4[2] = row_bcast<2>(a4); al4[3] = row_bcast<3>(a4);
    al4[4] = row_bcast<4>(a4); al4[5] = row_bcast<5>(a4);
    al4[6] = row_bcast<6>(a4); al4[7] = row_bcast<7>(a4);
    constexpr int NO = G * 8;
    float os[NO];
#pragma unroll
    for (int i = 0; i < NO; ++i) os[i] = o[i / 8][i % 8] * al4[i / 8];
#pragma unroll
    for (int i = 0; i < NO / 2; ++i) os[i] = swap_add<32>(os[i], os[i + NO / 2]);
#pragma unroll
    for (int i = 0; i < NO / 4; ++i) os[i] = swap_add<16>(os[i], os[i + NO / 4]);

    // cross-wave combine through LDS: row g16 now holds sums g16 * NO / 4 ... of its channels
    // (RUNS: two buffers in turn, as a wave may be a row ahead)
    auto& lds_o = lds_o_[RUNS ? turn : 0];
    auto& lds_ml = lds_ml_[RUNS ? turn : 0];
#pragma unroll
    for (int i = 0; i < NO / 4; ++i) {
        const int at = g16 * (NO / 4) + i;
        lds_o[wid][at / 8][dl * 8 + at % 8] = os[i];
    }
    if (lane < G) {
        lds_ml[wid][lane][0] = lsum > 0.0f ? mt4 : -INFINITY;
        lds_ml[wid][lane][1] = lsum;
    }
    __syncthreads();

    // 256 threads cover G*128 outputs, two channels each
    for (int idx = 2 * threadIdx.x; idx < G * DHEAD; idx += 2 * blockDim.x) {
        const int gh = idx / DHEAD;
        const int d = idx % DHEAD;
        float mt = -INFINITY;
#pragma unroll
        for (int w = 0; w < 4; ++w)
            if (lds_ml[w][gh][1] > 0.0f) mt = fmaxf(mt, lds_ml[w][gh][0]);
        float lt = 0.0f;
        float2 ot = {0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float lw = lds_ml[w][gh][1];
            const float sc = lw > 0.0f ? __expf(lds_ml[w][gh][0] - mt) : 0.0f;
            const float2 ow = *reinterpret_cast<const float2*>(&lds_o[w][gh][d]);
            lt += lw > 0.0f ? lw * sc : 0.0f;
            ot.x += lw > 0.0f ? ow.x * sc : 0.0f;
            ot.y += lw > 0.0f ? ow.y * sc : 0.0f;
        }
        *reinterpret_cast<float2*>(opart_row + gh * DHEAD + d) = ot;
        if (d == 0) {
            mlpart_row[gh * 2 + 0] = mt;
            mlpart_row[gh * 2 + 1] = lt;
            if (last) mlpart_row[(G + gh) * 2 + 1] = END_MARK;
        }
    }

    if (RUNS && left > 0) continue;
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
    return;
    }
}

// Combine split partials -> final output. Grid: B*Hq blocks of NG groups of 32 lanes; a
// group takes the splits s, s + NG, ..., a lane four channels. A small launch like this is
// its chain of loads, so a group's first two splits and all statistics are asked for
// together, and where the chip has room to spare (EARLY) even before the length says
// which of them exist: what a split past the end left is not looked at. Every wave works
// the common maximum and sum out for itself.
// RUNS: statistics and the first splits of two groups, which nearly always are there, are asked for
// before a mark says how many there are. Both launches, us, the splits counted from the lengths / by
// the mark: 64 of up to 300 tokens 22.9 / 20.8, 33 of up to 1500 39.9 / 38.5, 47 of up to 3000 76.7 /
// 74.5. Small launches would wait for it: decode steps of an 8B model, one sequence, 2926 us by marks, 2916 counted.
template <int G, bool EARLY, bool RUNS>
__global__ __launch_bounds__(EARLY ? 512 : 256) void decode_combine_kernel(
    const float* __restrict__ o_part, const float* __restrict__ ml_part,
    const int* __restrict__ seq_lens, uint32_t* __restrict__ out, int B, int Hk, int nsplit,
    int chunk_base, const int* __restrict__ slots) {
    constexpr int NG = EARLY ? 16 : 8;
    const int bq = blockIdx.x;
    const int Hq = Hk * G;
    const int b = bq / Hq;
    const int qh = bq % Hq;
    const int h = qh / G;
    const int gh = qh % G;
    const int lane = threadIdx.x & (WAVE - 1);
    const int grp = threadIdx.x >> 5, ch = (threadIdx.x & 31) * 4;
    size_t first = (size_t)(b * Hk + h) * nsplit * G + gh;
    const int n = seq_lens[b];
    if (!EARLY && !RUNS && slots && b > 0 && slots[b] == slots[0] && n == seq_lens[0] && n > 0 &&
        ml_part[first * 2 + 1] == COPY_MARK)
        first = (size_t)h * nsplit * G + gh;
    const float2* ml = reinterpret_cast<const float2*>(ml_part) + first;
    const float* op = o_part + first * DHEAD + ch;

    // the statistics of split `lane`, the first two splits of the own group, and how many exist
    const float2 none = {0.0f, 0.0f};
    float2 mine, mo[2];
    float4 ov[2];
    auto ask = [&](int i, int s) {
        mo[i] = ml[s * G];
        ov[i] = *reinterpret_cast<const float4*>(op + (size_t)s * G * DHEAD);
    };
    int ns = 0;
    if constexpr (RUNS) {
        auto look = [&]() {
            mine = ml[min(lane, nsplit - 1) * G];
            if (grp < 2) ask(0, min(grp, nsplit - 1));
        };
        look();
        if (slots && __any(lane == 0 && mine.y == COPY_MARK)) {
            first = (size_t)h * nsplit * G + gh;
            ml = reinterpret_cast<const float2*>(ml_part) + first;
            op = o_part + first * DHEAD + ch;
            look();
        }
        // the splits end at a mark or with the places
        for (int s0 = 0; n > 0 && s0 < nsplit; s0 += WAVE) {
            const bool end = s0 + lane >= nsplit || (s0 ? ml[(s0 + lane) * G] : mine).y == END_MARK;
            const uint64_t ends = __ballot(end);
            ns = s0 + (ends ? __builtin_ctzll(ends) : WAVE);
            if (ends) break;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int s = grp + NG * i;
            if (!(i == 0 && grp < 2) && s < ns) ask(i, s);
        }
    } else {
        ns = CEIL_DIV(n, decode_chunk(n, nsplit, chunk_base));
        // EARLY repeats the last split instead of a branch for each load
        mine = EARLY || lane < ns ? ml[(EARLY ? min(lane, nsplit - 1) : lane) * G] : none;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int s = EARLY ? min(grp + NG * i, nsplit - 1) : grp + NG * i;
            mo[i] = EARLY || s < ns ? ml[s * G] : none;
            ov[i] = EARLY || s < ns ? *reinterpret_cast<const float4*>(op + (size_t)s * G * DHEAD)
                                    : float4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }

    float mt = lane < ns && mine.y > 0.0f ? mine.x : -INFINITY;
    for (int s = lane + WAVE; s < ns; s += WAVE)
        if (ml[s * G].y > 0.0f) mt = fmaxf(mt, ml[s * G].x);
    mt = wave_reduce_max(mt);
    float lt = lane < ns && mine.y > 0.0f ? mine.y * __expf(mine.x - mt) : 0.0f;
    for (int s = lane + WAVE; s < ns; s += WAVE)
        if (ml[s * G].y > 0.0f) lt += ml[s * G].y * __expf(ml[s * G].x - mt);
    lt = wave_reduce_sum(lt);

    float4 ot = {0.0f, 0.0f, 0.0f, 0.0f};
    auto add = [&](const float2& m2, const float4& o4) {
        const float sc = __expf(m2.x - mt);
        ot.x += o4.x * sc;
        ot.y += o4.y * sc;
        ot.z += o4.z * sc;
        ot.w += o4.w * sc;
    };
#pragma unroll
    for (int i = 0; i < 2; ++i)
        if (grp + NG * i < ns && mo[i].y > 0.0f) add(mo[i], ov[i]);
    for (int s = grp + 2 * NG; s < ns; s += NG)
        if (ml[s * G].y > 0.0f)
            add(ml[s * G], *reinterpret_cast<const float4*>(op + (size_t)s * G * DHEAD));

    __shared__ __attribute__((aligned(16))) float red[NG][DHEAD];
    *reinterpret_cast<float4*>(&red[grp][ch]) = ot;
    __syncthreads();
    const int d = threadIdx.x;
    if (d >= DHEAD) return;
    float sum = 0.0f;
#pragma unroll
    for (int g = 0; g < NG; ++g) sum += red[g][d];
    const float res = (lt > 0.0f) ? sum / lt : 0.0f;
    reinterpret_cast<uint16_t*>(out)[(size_t)(b * Hq + qh) * DHEAD + d] = f32_to_bf16(res);
}

// Keys of the smallest split, by the (sequence, key head) pairs of the launch. Both
// launches, 8 key heads unless said, us with 64 / 128 / 256 / 512 keys: one sequence of
// 1151 tokens 9.9 / 10.6 / 11.4 / 14.4, 4 of 700 11.9 / 10.8 / 12.1 / 14.5, 13 of up to 900
// (4 key heads) 16.4 / 13.0 / 12.1 / 14.8, 8 of up to 1500 20.7 / 16.6 / 16.4 / 15.9, 16
// 32.7 / 25.9 / 24.1 / 25.8, 32 of up to 3000 84 / 75 / 65 / 63, 64 147 / 133 / 117 / 109
// (its cache rows alone take 82 at 6 TB/s), 64 of up to 300 30 / 26 / 23 / 22. Before rows
// merged by swaps and the combine asked ahead, the sizes in use took 13.0, 12.6, 15.0,
// 19.0, 26.3, 64.8, 112.8 and 24.0.
static int decode_chunk_base(int pairs) {
    return pairs <= 8 ? 64 : pairs <= 32 ? 128 : pairs <= 128 ? 256 : 512;
}

// Runs of a key head, 0 for splits of each sequence: under 512 (sequence, key head) pairs the host, which does
// not know the lengths, cannot tell where runs gain from where they and what a launch works out first cost
// more (both launches, us, splits / runs, 8 key heads, caches that no cache holds: 32 of up to 3000 tokens 66 /
// 57, 24 of 1500 in 32 35 / 32, but 32 of 700 21.8 / 26.6, 32 of 1000 28.4 / 30.5, 16 of 1000 18.8 / 20.4, 12 of 500
// 12.8 / 13.6).
static int decode_run_count(int B, int Hk, int nsplit) {
    return B * Hk < 512 || B > 4096 || nsplit < 2 ? 0 : max(1, 256 / Hk);
}

// Blocks of a key head: its runs, or the units that fewer than 8 * (runs + B) tiles make; rows that share
// pages take units that fit in
static int decode_run_blocks(int runs, int cb, int B) {
    return max(max(runs, 4 * B), 8 * (runs + B) * 64 / cb + B);
}

// Early loads pay while the launch is a few blocks (both launches, us: one sequence of 1151
// tokens 10.4 -> 9.9, 8 of up to 1500 16.9 -> 16.5) and cost where 2048 of them ask for
// splits that do not exist (64 of up to 300: 24.1 -> 25.0).
template <int G>
static void launch_combine(hipStream_t s, const void* o_part, const void* ml_part,
                           const void* seq_lens, void* out, int B, int Hk, int nsplit, int cb,
                           const void* slots, bool runs) {
#define LAUNCH_C(EARLY, RUNS)                                                                      \
    hipLaunchKernelGGL((decode_combine_kernel<G, EARLY, RUNS>), dim3(B * Hk * G),                  \
                       dim3((EARLY) ? 512 : 256), 0, s, (const float*)o_part, (const float*)ml_part, \
                       (const int*)seq_lens, (uint32_t*)out, B, Hk, nsplit, cb, (const int*)slots)
    if (runs) LAUNCH_C(false, true);
    else if (B * Hk <= 64) LAUNCH_C(true, false);
    else LAUNCH_C(false, false);
#undef LAUNCH_C
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

    if (fused) {
        hipError_t e = hipMemsetAsync(cnt_ws, 0, B * Hk * 4, (hipStream_t)stream);
        if (e != hipSuccess) return (int)e;
    }

    const int cb = decode_chunk_base(B * Hk);
    const int runs = fused ? 0 : decode_run_count(B, Hk, nsplit);
    if (runs) grid = dim3(Hk, decode_run_blocks(runs, cb, B));
#define LAUNCH_FORM(GV, FUSED, RUNS, ...)                                                      \
    hipLaunchKernelGGL((decode_attn_kernel<GV, FUSED, false, RUNS>), grid, block, 0,           \
                       (hipStream_t)stream, (const uint32_t*)q, (const uint32_t*)kc,           \
                       (const uint32_t*)vc, (const int*)block_table, (const int*)seq_lens,     \
                       (float*)o_part, (float*)ml_part, (unsigned*)cnt_ws, (uint32_t*)out, B,  \
                       Hk, max_blocks, block_shift, nsplit, cb, scale, qs2,                    \
                       (const uint32_t*)nullptr, (const uint32_t*)nullptr,                     \
                       (const float*)nullptr, (const float*)nullptr, (const int*)nullptr,      \
                       (uint32_t*)nullptr, (uint32_t*)nullptr, 0, 0, 0, ##__VA_ARGS__)
#define LAUNCH_G(GV)                                                                           \
    do {                                                                                       \
        if (fused) LAUNCH_FORM(GV, true, false);                                               \
        else if (runs) LAUNCH_FORM(GV, false, true, Runs{runs});                               \
        else LAUNCH_FORM(GV, false, false);                                                    \
        HIP_CHECK_LAUNCH();                                                                    \
        if (!fused) {                                                                          \
            launch_combine<GV>((hipStream_t)stream, o_part, ml_part, seq_lens, out, B, Hk,     \
                               nsplit, cb, nullptr, runs);                                     \
            HIP_CHECK_LAUNCH();                                                                \
        }                                                                                      \
    } while (0)

    switch (G) {
        case 1: LAUNCH_G(1); break;
        case 2: LAUNCH_G(2); break;
        case 4: LAUNCH_G(4); break;
        case 8: LAUNCH_G(8); break;
        default: return -102;
    }
#undef LAUNCH_G
#undef LAUNCH_FORM
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

    const int cb = decode_chunk_base(B * Hk);
    // few blocks wait for their slowest, which is then a copy looked at twice
    const int copies = B * Hk > 64;
    const int runs = decode_run_count(B, Hk, nsplit);
    // rows that may be copies follow the runs
    if (runs) grid = dim3(Hk, decode_run_blocks(runs, cb, B) + copies * (B - 1));
#define LAUNCH_FORM(GV, RUNS, ...)                                                             \
    hipLaunchKernelGGL((decode_attn_kernel<GV, false, true, RUNS>), grid, block, 0,            \
                       (hipStream_t)stream, (const uint32_t*)q, (const uint32_t*)kc,           \
                       (const uint32_t*)vc, (const int*)block_table, (const int*)seq_lens,     \
                       (float*)o_part, (float*)ml_part, (unsigned*)nullptr, (uint32_t*)out, B, \
                       Hk, max_blocks, block_shift, nsplit, cb, scale, q_stride / 2,           \
                       (const uint32_t*)kin, (const uint32_t*)vin, (const float*)cos_t,        \
                       (const float*)sin_t, (const int*)slots, (uint32_t*)kc, (uint32_t*)vc,   \
                       k_stride / 2, v_stride / 2, copies, ##__VA_ARGS__)
#define LAUNCH_GR(GV)                                                                          \
    do {                                                                                       \
        if (runs) LAUNCH_FORM(GV, true, Runs{runs});                                           \
        else LAUNCH_FORM(GV, false);                                                           \
        HIP_CHECK_LAUNCH();                                                                    \
        launch_combine<GV>((hipStream_t)stream, o_part, ml_part, seq_lens, out, B, Hk, nsplit, \
                           cb, copies ? slots : nullptr, runs);                                \
        HIP_CHECK_LAUNCH();                                                                    \
    } while (0)

    switch (G) {
        case 1: LAUNCH_GR(1); break;
        case 2: LAUNCH_GR(2); break;
        case 4: LAUNCH_GR(4); break;
        case 8: LAUNCH_GR(8); break;
        default: return -102;
    }
#undef LAUNCH_GR
#undef LAUNCH_FORM
    return 0;
}

// Whether a launch of as many (sequence, key head) pairs takes the projection's planes: up to 64 of them,
// where there are neither runs nor copies of the first row
extern "C" int oa_attention_decode_takes_parts(int B, int Hq, int Hk, int D) {
    const int G = Hk > 0 && Hq % Hk == 0 ? Hq / Hk : 0;
    return D == DHEAD && (G == 1 || G == 2 || G == 4 || G == 8) && (int64_t)B * Hk <= 64;
}

// oa_attention_decode_rope of a projection that is still its planes part [splits, B, (Hq + 2 Hk) * D]
extern "C" int oa_attention_decode_parts(
    void* stream, const void* part, int splits, void* kc, void* vc, const void* block_table, const void* seq_lens,
    const void* cos_t, const void* sin_t, const void* slots, void* o_part, void* ml_part, void* out, int B, int Hq,
    int Hk, int D, int max_blocks, int block_size, int nsplit, float scale) {
    if (B < 1 || splits < 1 || nsplit < 1 || !oa_attention_decode_takes_parts(B, Hq, Hk, D)) return -100;
    if ((block_size & (block_size - 1)) != 0) return -101;
    if ((uintptr_t)part % 16 != 0) return -103;
    int block_shift = 0;
    while ((1 << block_shift) < block_size) ++block_shift;
#define LAUNCH_P(GV)                                                                                              \
    do {                                                                                                          \
        hipLaunchKernelGGL((decode_attn_kernel<GV, false, true, false>), dim3(B * Hk, nsplit), dim3(256), 0,       \
                           (hipStream_t)stream, (const uint32_t*)nullptr, (const uint32_t*)kc,                    \
                           (const uint32_t*)vc, (const int*)block_table, (const int*)seq_lens, (float*)o_part,    \
                           (float*)ml_part, (unsigned*)nullptr, (uint32_t*)out, B, Hk, max_blocks, block_shift,   \
                           nsplit, decode_chunk_base(B * Hk), scale, 0, (const uint32_t*)nullptr,                 \
                           (const uint32_t*)nullptr, (const float*)cos_t, (const float*)sin_t, (const int*)slots, \
                           (uint32_t*)kc, (uint32_t*)vc, 0, 0, 0,                                                 \
                           (Planes{(const float*)part, splits, (int64_t)B * (Hq + 2 * Hk) * DHEAD}));             \
        HIP_CHECK_LAUNCH();                                                                                       \
        launch_combine<GV>((hipStream_t)stream, o_part, ml_part, seq_lens, out, B, Hk, nsplit,                    \
                           decode_chunk_base(B * Hk), nullptr, false);                                            \
        HIP_CHECK_LAUNCH();                                                                                       \
    } while (0)
    switch (Hq / Hk) {
        case 1: LAUNCH_P(1); break;
        case 2: LAUNCH_P(2); break;
        case 4: LAUNCH_P(4); break;
        default: LAUNCH_P(8); break;
    }
#undef LAUNCH_P
    return 0;
}
