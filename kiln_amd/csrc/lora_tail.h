// The low-rank term the small-M kernels add where they store a tile (gfx950 only).
#pragma once
#include <type_traits>

#include "device_common.h"
#include "launch.h"

namespace kiln {

// Optional low-rank term of the result: y += T * B_cat^T, where T = bf16 [M, rp] is the scaled
// projection of the activations onto the stacked adapters (columns r_total ... rp - 1 zero, rp a
// multiple of 16) and B_cat = bf16 [N, r_total] (crates/kiln-model/src/lora_loader.rs:213-232,
// added unfused at forward.rs:2932-2939).  rp == 0: none.
struct LoraTail {
    const uint16_t *t;
    const uint16_t *b;
    int r_total;
    int rp;
    int slices;    // T = [slices][t_rows][rp]: K slices of the projection, each rounded on its own
    int t_rows;
};

// v = rows row0 + 4 (lane / 16) ... + 3 of column lane % 16 of tile tt, in the accumulator layout.
// rp <= 64: two steps of 32 rank columns at most.  Everything a chunk of eight slices needs is
// requested before the first product (one memory round trip instead of one per step: the operands
// come from L2 or beyond, 1...2 us away, and this sits at the very end of the launch).
[[maybe_unused]] __device__ __forceinline__ void lora_add(f32x4 &v, const LoraTail &lo, int row0, int M, int tt,
                                                          int lane) {
    const int kq = lane >> 4, c = lane & 15;
    int row = row0 + c;
    row = row < M ? row : M - 1;  // rows past M: any finite operand, the products are never stored
    const uint16_t *tp = lo.t + (size_t)row * lo.rp;
    const uint16_t *bp = lo.b + (size_t)(tt * kTileN + c) * lo.r_total;
    u32x4 tb[2];
#pragma unroll
    for (int js = 0; js < 2; ++js) {
        const int j8 = 32 * js + 8 * kq;  // this lane's 8 rank columns of step js
        tb[js] = u32x4{0u, 0u, 0u, 0u};
        if ((lo.r_total & 7) == 0) {
            if (j8 < lo.r_total) tb[js] = *reinterpret_cast<const u32x4 *>(bp + j8);
        } else {
            uint32_t e[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) e[i] = (j8 + i < lo.r_total) ? (uint32_t)bp[j8 + i] : 0u;
            tb[js] = u32x4{e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16)};
        }
    }
    for (int z0 = 0; z0 < lo.slices; z0 += 8) {  // eight slices requested at a time
        u32x4 ta[2][8];
#pragma unroll
        for (int js = 0; js < 2; ++js) {
            const int j8 = 32 * js + 8 * kq;
#pragma unroll
            for (int zi = 0; zi < 8; ++zi) {
                ta[js][zi] = u32x4{0u, 0u, 0u, 0u};
                if (j8 < lo.rp && z0 + zi < lo.slices)
                    ta[js][zi] = *reinterpret_cast<const u32x4 *>(tp + (size_t)(z0 + zi) * lo.t_rows * lo.rp + j8);
            }
        }
#pragma unroll
        for (int js = 0; js < 2; ++js)
#pragma unroll
            for (int zi = 0; zi < 8; ++zi)
                if (32 * js < lo.rp && z0 + zi < lo.slices)
                    v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ta[js][zi]),
                                                                __builtin_bit_cast(bf16x8, tb[js]), v, 0, 0, 0);
    }
}

// The same term with its operands in LDS: T whole ([slices][t_rows][rp], t_rows = M) and the
// r_total-wide rows of B_cat of the block's columns (tile ti of the block starts at row 16 ti);
// r_total % 8 == 0.  v = rows 4 (lane / 16) ... + 3 of column lane % 16 of the tile.
__device__ __forceinline__ void lora_add_from_lds(f32x4 &v, const LoraTail &lo, const unsigned char *t_lds,
                                                  const unsigned char *b_lds, int ti, int M, int lane) {
    const int kq = lane >> 4, c = lane & 15;
    const int row = c < M ? c : M - 1;  // rows past M: any finite operand, the products are never stored
    for (int j0 = 0; j0 < lo.rp; j0 += 32) {
        const int j8 = j0 + 8 * kq;  // this lane's 8 rank columns
        u32x4 tb = {0u, 0u, 0u, 0u};
        if (j8 < lo.r_total) tb = *reinterpret_cast<const u32x4 *>(b_lds + ((ti * kTileN + c) * lo.r_total + j8) * 2);
        for (int z = 0; z < lo.slices; ++z) {
            u32x4 ta = {0u, 0u, 0u, 0u};
            if (j8 < lo.rp) ta = *reinterpret_cast<const u32x4 *>(t_lds + ((z * lo.t_rows + row) * lo.rp + j8) * 2);
            v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ta), __builtin_bit_cast(bf16x8, tb), v, 0,
                                                        0, 0);
        }
    }
}

// A value in a scalar register of its own (a choice between an argument's members would otherwise become one between their
// addresses, in scratch memory).
template <class V>
__device__ __forceinline__ V scalar(V v) {
    asm("" : "+s"(v));
    return v;
}
// The adapters of projections that run as one GEMM, where they lie: side i has A = bf16 [ranks, K] and B = bf16
// [rows, ranks] of its own, ranks a multiple of 8, and the columns from col[i] on of the stacked rank axis.  Its rows of B
// are the GEMM's columns from first[i] on; interleaved, those of every 16-column tile from first[i] (0: gate, 8: up) on,
// eight of them.  Columns of no side have no term.  What it saves is launches, which bound these calls: stacking took one
// of 3.4 us in front of every fused call, and q | k | v with two adapters each, six together, another of 5 us for the
// projection, which the stacked form takes inside for four at most.  (A layer at 11 rows, two adapters of rank 8 on each
// projection, 2560 / 9216 wide: 41.2 -> 33.1 us, four launches instead of seven.  On the mid-M kernel, six launches -> four:
// at 20 / 50 / 100 rows 52.4 -> 46.7 / 63.0 -> 57.0 / 87.7 -> 82.0 us; 1536 / 5120 wide 47.3 -> 42.0 / 48.6 -> 44.0 / 58.7 -> 53.0.)
// (The gate | up launch alone then took 10.6 us at 11 rows where it took 9.2 behind the launch that stacked: its adapter
// wavefront waited for the rows of B before it looked at the producers' flags, which it does no longer.)
struct LoraSides {
    const uint16_t *a[kMaxAdapterSides];
    const uint16_t *b[kMaxAdapterSides];
    int col[kMaxAdapterSides + 1];   // past the last side: r_total
    int first[kMaxAdapterSides];
    int rows[kMaxAdapterSides];
    int count;
    int interleaved;
};
// the row of A of a rank column
__device__ __forceinline__ const uint16_t *side_a_row(const LoraSides &s, int rank, int K) {
    const uint16_t *base = s.a[0];
    int from = 0;
#pragma unroll
    for (int i = 1; i < kMaxAdapterSides; ++i)
        if (i < s.count && rank >= s.col[i]) {
            base = s.a[i];
            from = s.col[i];
        }
    return base + (size_t)(rank - from) * K;
}
// Where eight rank columns from j8 on (a multiple of 8) of a column's row of B lie; not live: no side's.  Found without a branch.
struct SideUnit {
    const void *at;
    bool live;
};
__device__ __forceinline__ SideUnit side_b_unit(const LoraSides &s, int column, int j8) {
    uint64_t at = reinterpret_cast<uint64_t>(s.b[0]);
    bool live = false;
#pragma unroll
    for (int i = 0; i < kMaxAdapterSides; ++i) {
        const int row = s.interleaved ? (column >> 4) * 8 + (column & 7) : column - s.first[i], ranks = s.col[i + 1] - s.col[i];
        const bool in_side = s.interleaved ? (column & 8) == s.first[i] : (uint32_t)row < (uint32_t)s.rows[i];
        const bool mine = in_side & ((uint32_t)(j8 - s.col[i]) < (uint32_t)ranks);  // (never of a side past the last: no ranks)
        const uint64_t b = scalar(reinterpret_cast<uint64_t>(s.b[i]));
        at = mine ? b + (uint64_t)(uint32_t)(row * ranks + j8 - s.col[i]) * 2 : at;
        live |= mine;
    }
    return SideUnit{reinterpret_cast<const void *>(at), live};
}
inline LoraSides lora_sides(const AdapterSides *h) {
    LoraSides s{};
    s.count = h->count;
    s.interleaved = h->interleaved;
    for (int i = 0; i < h->count; ++i) {
        s.a[i] = (const uint16_t *)h->a[i];
        s.b[i] = (const uint16_t *)h->b[i];
        s.first[i] = h->first[i];
        s.rows[i] = h->rows[i];
        s.col[i + 1] = s.col[i] + h->ranks[i];
    }
    for (int i = h->count; i < kMaxAdapterSides; ++i) s.col[i + 1] = s.col[i];
    return s;
}

// The projection T computed inside the launch that adds it, by `producers` extra blocks at the
// front of the grid (one K slice each) while the other blocks stream their weights.  A producer
// writes its slice of T with device-scope stores, waits until they are acknowledged and raises
// its flag; the blocks that add the term look at the flags through one wavefront (while the
// others sum their tiles) and read T with ordinary loads once the flags are up (no cache on
// their die has seen those lines since the launch began).  The flag words and the reader counts
// live in workspace that is all zero between launches: every adding block counts itself after
// its look, and the last one to do so zeroes the words.  Hundreds of blocks looking at one
// address, or counting on one, are served one after the other (measured: 231 single polls of one
// 64-byte line, every flag already up, took up to 4 us, and as long again for their 231 atomic
// adds on one counter): the flags therefore exist kLoraFoldReplicas times, 4 KiB apart, block b
// looks at and counts on replica b % kLoraFoldReplicas, and whoever completes a replica's count
// counts once more on a top word.  producers == 0: T comes from a launch of its own.
struct LoraFold {
    const uint16_t *a_cat;   // bf16 [r_total, K]: the adapters' A matrices stacked along rows
    uint16_t *t;             // where the producers write T: [producers][t_rows][rp] bf16
    unsigned *flags;         // kLoraFoldReplicas x kLoraFoldReplicaWords words: per replica one flag per producer,
                             // then the replica's reader count; the top count behind that in replica 0
    int producers;           // K slices of the projection
    int steps_per_slice;     // 32-value steps of K per slice
    int consumers;           // blocks that add the term
    // exclusive end column of adapter i on the stacked rank axis (r_total past the last adapter) and its
    // scale (0 past the last); plain members, not arrays: an indexed kernel argument is copied to scratch memory
    int e0, e1, e2, e3;      // (four adapters at most: every member is a scalar register for the whole kernel)
    float s0, s1, s2, s3;
};
// ... of unstacked adapters, which a_cat, the tail's b and the four above do not describe.  Instances of their own: with
// both forms in one kernel the stacked one lost 0.1 to 0.5 us a launch to the other's registers.
struct LoraSidesFold : LoraFold {
    LoraSides sides;
    int ends[8];             // read with constant indices only
    float scales[8];
};
// The adapters of a call whose blocks project x onto them by themselves (own_tiles): the sides of LoraSides, one for a
// stacked set, prepared so that a row or a unit is found without a branch.  A side that is absent has no columns.
// (Plain members, not arrays: what is picked from an array by a condition goes through scratch memory.)
static_assert(kMaxAdapterSides == 3, "three members of each kind below");
struct OwnSidesA {
    uint64_t a0, a1, a2;           // less col[i] rows of A: the row of a stacked rank column is that many rows on
    int col1, col2, col3;          // the first stacked rank column of side 1, 2, past the last one
    int first0, first1, first2;    // the columns of the GEMM that have a term of the side lie in [first, end)
    int end0, end1, end2;
    int unused;
};
struct OwnSidesB {
    uint64_t b0, b1, b2;
    int col1, col2, col3;
    int first0, first1, first2;    // columns whose masked index lies in [first, first + span) are the side's
    int span0, span1, span2;
    int key_mask, row_shift, low_mask;  // interleaved 8, 1, 7: row = 8 (column / 16) + column % 8; else -1, 0, 15 ...
    int row_counts_from_first;     // ... and 1: less the side's first column
    int unused;
};
struct OwnScales {
    int ends[8];                   // read with constant indices only
    float scales[8];
};
struct OwnArgs {
    OwnSidesA a;
    OwnSidesB b;
    OwnScales scales;
};
struct LoraOwnFold : LoraFold {
    OwnArgs own;
};
// On the device, free of branches: it runs while the first weights are in flight to registers.
struct OwnWindow {  // the stacked rank columns that the block's columns have a term of
    int lo, ranks;
};
[[maybe_unused]] __device__ __forceinline__ OwnWindow own_window(const OwnSidesA &s, int first_column, int end_column) {
    const bool here0 = (s.first0 < end_column) & (s.end0 > first_column), here1 = (s.first1 < end_column) & (s.end1 > first_column),
               here2 = (s.first2 < end_column) & (s.end2 > first_column);
    int lo = here2 ? s.col2 : s.col3, hi = here0 ? s.col1 : 0;
    lo = here1 ? s.col1 : lo;
    lo = here0 ? 0 : lo;
    hi = here1 ? s.col2 : hi;
    hi = here2 ? s.col3 : hi;
    lo = min(lo, hi);
    return OwnWindow{lo, hi - lo};
}
// the row of A of a stacked rank column
[[maybe_unused]] __device__ __forceinline__ const char *own_a_row(const OwnSidesA &s, int rank, uint32_t row_bytes) {
    const uint64_t a1 = scalar(s.a1), a2 = scalar(s.a2);
    uint64_t base = scalar(s.a0);
    base = rank >= s.col1 ? a1 : base;
    base = rank >= s.col2 ? a2 : base;
    return reinterpret_cast<const char *>(base + (uint64_t)(uint32_t)rank * row_bytes);
}
// Where four rank columns from `rank` on of a column's row of B_cat lie; false (and an address that can be read): no term.
[[maybe_unused]] __device__ __forceinline__ bool own_b_unit(const OwnSidesB &s, int column, int rank, const void **at) {
    const int key = column & s.key_mask, row = ((column & ~15) >> s.row_shift) + (column & s.low_mask);
    uint64_t p = scalar(s.b0);
    int from = 0;
    bool live = false;
    auto side = [&](uint64_t b, int first, int span, int col, int end) {
        const int width = end - col;
        const bool mine = ((uint32_t)(key - first) < (uint32_t)span) & ((uint32_t)(rank - col) < (uint32_t)width);
        p = mine ? b : p;
        // (of 24 bits: cheap enough that the compiler forms it for every side instead of behind a branch)
        const int at_unit = __mul24(row - __mul24(first, s.row_counts_from_first), width) + rank - col;
        from = mine ? at_unit : from;
        live |= mine;
    };
    side(scalar(s.b0), s.first0, s.span0, 0, s.col1);
    side(scalar(s.b1), s.first1, s.span1, s.col1, s.col2);
    side(scalar(s.b2), s.first2, s.span2, s.col2, s.col3);
    *at = reinterpret_cast<const void *>(p + (uint64_t)(uint32_t)from * 2);
    return live;
}
template <class Args>  // DecodeArgs, MidArgs
OwnArgs own_args(const Args &d) {
    const AdapterSides &h = *d.lora_sides;
    const bool all = !own_blocks_end_with_sides(h, d.lora_adapters, d.M);
    uint64_t a[3] = {}, b[3] = {};
    int col[4] = {}, first[3] = {}, end[3] = {}, key[3] = {}, span[3] = {};
    for (int i = 0; i < kMaxAdapterSides; ++i) {
        col[i + 1] = col[i];
        if (i >= h.count) continue;
        a[i] = reinterpret_cast<uint64_t>(h.a[i]) - (uint64_t)col[i] * d.K * 2;
        b[i] = reinterpret_cast<uint64_t>(h.b[i]);
        first[i] = all ? 0 : h.first[i];
        end[i] = all ? d.N : h.first[i] + h.rows[i];
        key[i] = h.first[i];
        span[i] = h.interleaved ? 8 : h.rows[i];
        col[i + 1] += h.ranks[i];
    }
    OwnArgs o{};
    o.a = OwnSidesA{a[0], a[1], a[2], col[1], col[2], col[3], first[0], first[1], first[2], end[0], end[1], end[2], 0};
    o.b = OwnSidesB{b[0], b[1], b[2], col[1], col[2], col[3], key[0], key[1], key[2], span[0], span[1], span[2],
                    h.interleaved ? 8 : -1, h.interleaved ? 1 : 0, h.interleaved ? 7 : 15, h.interleaved ? 0 : 1, 0};
    for (int i = 0; i < 8; ++i) {
        o.scales.ends[i] = d.lora_ends[i];
        o.scales.scales[i] = d.lora_scales[i];
    }
    return o;
}
constexpr int kLoraFoldMaxProducers = 16;
constexpr int kLoraSidesMaxAdapters = 8;
constexpr int kLoraFoldStepsPerWave = 12;  // 32-value steps of K one producer wavefront takes, at most
constexpr int kLoraFoldReplicas = 16;
constexpr int kLoraFoldReplicaWords = 1024;                  // 4 KiB from one replica to the next
constexpr int kLoraFoldCountWord = kLoraFoldMaxProducers;    // a replica's reader count
constexpr int kLoraFoldTopWord = kLoraFoldMaxProducers + 1;  // in replica 0: completed replicas
constexpr size_t kLoraFoldFlagBytes = (size_t)kLoraFoldReplicas * kLoraFoldReplicaWords * sizeof(unsigned);
constexpr int kLoraFoldSpinLimit = 1 << 20;

// One producer block: slice `slice` of T = scale(j) * x * a_cat^T for up to 16 rows of x (bf16 [M, K]),
// rounded to bf16 (crates/kiln-model/src/lora_loader.rs:213-232, the first product, with the
// adapter scale folded in before the rounding).  Wavefront w takes rank tile w % JT and every
// Q-th step of the slice from w / JT on (JT = rp / 16 rank tiles, Q = nw / JT; nw >= JT); the Q
// parts of a tile meet in LDS (nw KiB) and are added in ascending order.  Every wavefront of the
// block must call this (two barriers inside).
template <class Fold>
__device__ __forceinline__ void lora_project_slice(const uint16_t *__restrict__ X, const Fold &fold,
                                                   const LoraTail &lo, int M, int K, int slice,
                                                   unsigned char *lds, int wave, int lane, int nw) {
    const int JT = lo.rp >> 4, Q = nw / JT;
    const int steps = K >> 5, s0 = slice * fold.steps_per_slice, s1 = min(steps, s0 + fold.steps_per_slice);
    const int r = lane & 15, kq = lane >> 4;
    const int jt = wave % JT, q = wave / JT;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (q < Q) {
        const int rank = jt * 16 + r;
        const uint16_t *xp = X + (size_t)min(r, M - 1) * K + kq * 8;
        const uint16_t *ap;
        if constexpr (std::is_same_v<Fold, LoraSidesFold>) ap = side_a_row(fold.sides, min(rank, lo.r_total - 1), K) + kq * 8;
        else ap = fold.a_cat + (size_t)min(rank, lo.r_total - 1) * K + kq * 8;
        const bool live = rank < lo.r_total;  // padding columns of T are zero
        // four steps requested at a time (more in flight would raise the whole kernel's register count,
        // and with it the launch cost of calls without adapters: measured +0.45 us at 97 instead of 82)
        for (int i0 = 0; i0 < kLoraFoldStepsPerWave; i0 += 4) {
            u32x4 xa[4], aa[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int st = s0 + q + (i0 + i) * Q;
                xa[i] = aa[i] = u32x4{0u, 0u, 0u, 0u};
                if (st < s1) {
                    xa[i] = *reinterpret_cast<const u32x4 *>(xp + (size_t)st * 32);
                    if (live) aa[i] = *reinterpret_cast<const u32x4 *>(ap + (size_t)st * 32);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xa[i]),
                                                              __builtin_bit_cast(bf16x8, aa[i]), acc, 0, 0, 0);
            if (s0 + q + (i0 + 4) * Q >= s1) break;
        }
    }
    f32x4 *parts = reinterpret_cast<f32x4 *>(lds);
    parts[wave * 64 + lane] = acc;
    __syncthreads();
    if (wave < JT) {  // rows 4 (lane / 16) ... + 3 of rank column 16 wave + lane % 16
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
        for (int q2 = 0; q2 < Q; ++q2) sum += parts[(wave + q2 * JT) * 64 + lane];
        const int j = wave * 16 + r;
        // the scale of the first adapter whose columns end behind j
        float sc = 0.f;
        if constexpr (std::is_same_v<Fold, LoraSidesFold>) {
#pragma unroll
            for (int i = kLoraSidesMaxAdapters - 1; i >= 0; --i) sc = j < fold.ends[i] ? fold.scales[i] : sc;
        } else {
            sc = j < fold.e3 ? fold.s3 : sc;
            sc = j < fold.e2 ? fold.s2 : sc;
            sc = j < fold.e1 ? fold.s1 : sc;
            sc = j < fold.e0 ? fold.s0 : sc;
        }
        uint16_t *tz = fold.t + (size_t)slice * lo.t_rows * lo.rp;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // two neighbouring columns per 32-bit device-scope store (even lanes)
            const uint32_t mine = f32_to_bf16_bits(sum[i] * sc);
            const uint32_t next = (uint32_t)__shfl_xor((int)mine, 1, 64);
            const int row = 4 * kq + i;
            if ((lane & 1) == 0 && row < M)
                __hip_atomic_store(reinterpret_cast<uint32_t *>(tz + (size_t)row * lo.rp + j), mine | (next << 16),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // this wavefront's part of T has reached memory
    __syncthreads();
    if (wave == 0 && lane < kLoraFoldReplicas)
        __hip_atomic_store(fold.flags + lane * kLoraFoldReplicaWords + slice, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A block that adds the term (the `consumer`-th of them), one wavefront of it: wait until every
// producer has raised its flag.  The bound is never reached in a working launch.
__device__ __forceinline__ int lora_fold_wait(const LoraFold &fold, int consumer, int lane) {
    const unsigned *mine = fold.flags + (consumer % kLoraFoldReplicas) * kLoraFoldReplicaWords;
    int spins = 0;
    for (; spins < kLoraFoldSpinLimit; ++spins) {
        unsigned f = 1u;
        if (lane < fold.producers) f = __hip_atomic_load(mine + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__builtin_amdgcn_ballot_w64(f == 0u) == 0) break;
        __builtin_amdgcn_s_sleep(4);
    }
    return spins;  // polls that came back without every flag
}

// The same wavefront, after its look: count this block on its replica; the block that completes a
// replica counts on the top word, and the one that completes that has seen every other block
// past its look at the flags and zeroes flags and counts for the next launch.
__device__ __forceinline__ void lora_fold_done(const LoraFold &fold, int consumer, int lane) {
    const int replica = consumer % kLoraFoldReplicas;
    const unsigned quota = (unsigned)(fold.consumers - replica + kLoraFoldReplicas - 1) / kLoraFoldReplicas;
    const unsigned replicas = (unsigned)min(fold.consumers, kLoraFoldReplicas);
    unsigned before = 0;
    if (lane == 0)
        before = __hip_atomic_fetch_add(fold.flags + replica * kLoraFoldReplicaWords + kLoraFoldCountWord, 1u,
                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    before = (unsigned)__builtin_amdgcn_readfirstlane((int)before);
    if (before != quota - 1u) return;
    if (lane == 0)
        before = __hip_atomic_fetch_add(fold.flags + kLoraFoldTopWord, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    before = (unsigned)__builtin_amdgcn_readfirstlane((int)before);
    if (before != replicas - 1u) return;
    if (lane <= kLoraFoldTopWord)
        for (int r = 0; r < kLoraFoldReplicas; ++r)
            __hip_atomic_store(fold.flags + r * kLoraFoldReplicaWords + lane, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

inline LoraTail lora_tail(const DecodeArgs &a) {
    LoraTail lo{};
    if (a.r_total > 0) {
        lo.t = (const uint16_t *)a.lora_t;
        lo.b = (const uint16_t *)a.lora_b;
        lo.r_total = a.r_total;
        lo.rp = (a.r_total + 15) / 16 * 16;
        lo.slices = a.lora_slices;
        lo.t_rows = a.lora_rows;
    }
    return lo;
}

}  // namespace kiln
