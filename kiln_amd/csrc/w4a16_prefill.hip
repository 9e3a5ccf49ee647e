// Large-M (prefill) W4A16 GEMM kernel for gfx950.
//
// Replaces the m > 16 arm of the reference dispatcher and kernel
// (crates/kiln-marlin-gemm/csrc/marlin_kernel.cu:754-763, :784-816, :189-700).
// This regime is a dense contraction bound by the bf16 matrix cores.
//
// Block = 4 wavefronts side by side, block tile 128 (or 64) rows x 256 columns,
// wavefront tile 128 x 64 = 4 x 2 tiles of v_mfma_f32_32x32x16_bf16 (128
// accumulator registers, two wavefronts per SIMD).  Per 32 rows of K:
//   * a 128 x 32 bf16 tile of A goes global -> LDS with direct 128-bit loads
//     (no registers, no VALU) into a ring of four stages, four stages ahead
//     of the products, one barrier per stage, stored with an XOR swizzle so
//     that fragment reads are bank-conflict free;
//   * each wavefront reads its 64 columns of packed weights straight from
//     global memory (four 128-bit loads per lane and 128-row group, prefetched
//     one group ahead) and expands the codes in registers: weights never touch
//     LDS, and each expanded fragment feeds four products.
// Group scales are applied in f32 by a running rescale of the accumulator (one
// multiply per accumulator register and group): after group g it holds
// (partial result) / scale(g); the step to the next group multiplies by
// scale(g) / scale(g+1).  No second accumulator set is needed, and scales are
// never rounded into the weights.
// The B operand carries 136 + d (d = code - 8).  The surplus
// 136 * sum_k(a) * scale is removed at the end by a short extra contraction
// over "extension" operands: per (row, group) the value c = -136 * sum_k a,
// split exactly into three bf16 terms by the pre-pass kernel below, times the
// group scale split exactly into two bf16 terms; six exact products per group
// accumulate c * scale into the result (about 5 % extra matrix work).
// Launches of several rounds of 128-row blocks, with adapters or without, and of tiles that leave no
// compute units for the row sums, take c as f32 and add it where a group begins, in the rescale's
// multiplication (INC below): no extra matrix work.  Where a compute unit gets one block at most, the
// block has a second set of wavefronts for the other half of its K (WK below).
#include <climits>
#include <type_traits>

#include "device_common.h"
#include "launch.h"
#include "lora_tail.h"
#include "lora_project.h"
#include "async_loads.h"

namespace kiln {

namespace {

constexpr int kAStages = 4;

// c[m][g] = -136 * sum_{k in group g} a[m][k], group-major ([g][m]), for instances of the kernel that add it at every
// change of group: as f32 (PLAIN); for the others split into bf16 hi/mid/lo and stored as the 8-slot extension
// operand [hi, hi, mid, mid, lo, lo, 0, 0].
template <bool PLAIN>
__global__ __launch_bounds__(256) void w4a16_prefill_rowsum_kernel(const uint16_t *__restrict__ A,
                                                                 u32x4 *__restrict__ aext, int M, int K) {
    const int G = K / kGroupK;
    const int item = blockIdx.x * 16 + (threadIdx.x >> 4);  // (row, group), 16 lanes each
    const int sub = threadIdx.x & 15;
    if (item >= M * G) return;
    const int row = item / G, g = item - row * G;
    float sum = sum_bf16x8(*reinterpret_cast<const u32x4 *>(A + (size_t)row * K + (size_t)g * kGroupK + sub * 8));
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 16);
    if (sub == 0) store_row_sum(aext, (size_t)g * M + row, sum, PLAIN);  // group-major: the 32 rows of a half-wavefront are contiguous
}

template <int RB, bool PLAIN>
__global__ __launch_bounds__(256) void w4a16_lora_project_kernel(const uint16_t *__restrict__ X,
                                                                const uint16_t *__restrict__ a_cat,
                                                                uint16_t *__restrict__ T, int M, int K, int r_total,
                                                                int RP, int steps_per_slice, LoraScales ls,
                                                                float *partial, int *counters, u32x4 *aext) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    lora_project_block<RB, PLAIN>(lds, X, a_cat, T, M, K, r_total, RP, steps_per_slice, ls, partial, counters, aext,
                                  blockIdx.x, blockIdx.y, gridDim.y, nullptr);
}

typedef __attribute__((address_space(3))) void *lds_ptr_t;

// 128-bit direct global -> LDS load: lane i's 16 bytes land at lds_addr + 16 i.
// Written as inline asm on purpose.  Through the compiler's builtin, every
// later LDS read is preceded by a wait for *all* outstanding loads (the
// compiler cannot tell which ring slot a direct load targets), which would
// serialise the pipeline; completion is tracked by the explicit s_waitcnt
// before each barrier instead.  Only addresses enter the asm, never loaded data.
// Plain global loads issued the same way (the compiler counts only the loads it
// knows about, so a compiler-tracked load consumed while asm loads are in
// flight would drain the whole queue).  The results may be used only after an
// explicit s_waitcnt that covers them, followed by pin() on the registers.
__device__ __forceinline__ u32x4 async_load_b128(const u32x4 *p) {
    u32x4 v;
    asm volatile("global_load_dwordx4 %0, %1, off" : "=&v"(v) : "v"(p) : "memory");
    return v;
}
__device__ __forceinline__ uint32_t async_load_u16(const uint16_t *p) {
    uint32_t v;
    asm volatile("global_load_ushort %0, %1, off" : "=&v"(v) : "v"(p) : "memory");
    return v;
}
// Orders every later use of v after this point (and hence after the preceding s_waitcnt).
__device__ __forceinline__ void pin(u32x4 &v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void pin(uint32_t &v) { asm volatile("" : "+v"(v)); }

// immediate of s_waitcnt for vmcnt(n), other counters unconstrained
constexpr int vmcnt_imm(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }

__device__ __forceinline__ void direct_load_b128(const void *gptr, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                 :
                 : "v"(gptr), "s"(lds_addr)
                 : "memory", "m0");
}

// Probe builds only (-DKILN_PREFILL_TIMELINE): wall-clock stamps per block.
#ifdef KILN_PREFILL_TIMELINE
__device__ long long *g_timeline;
#define KILN_TL(i)                                                                              \
    do {                                                                                        \
        if (threadIdx.x == 0) {                                                                 \
            g_timeline[(size_t)blockIdx.x * 8 + (i)] = __builtin_amdgcn_s_memrealtime();        \
            if ((i) < 2) g_timeline[(size_t)blockIdx.x * 8 + 6 + (i)] = __builtin_amdgcn_s_memtime(); \
        }                                                                                       \
    } while (0)
#else
#define KILN_TL(i) \
    do {           \
    } while (0)
#endif

// v from the lane selected by a data-parallel-primitive control word (no LDS traffic)
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}

// Two values of a lane's column in neighbouring rows -> two bf16 values of neighbouring columns in one row: even lanes
// get the first row's, odd lanes the second's (each pair of lanes swaps one value).
__device__ __forceinline__ uint32_t neighbours_of_a_row(float first, float second, int lane) {
    const uint32_t own = f32_to_bf16_bits(first) | ((uint32_t)f32_to_bf16_bits(second) << 16);
    const uint32_t other = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)own, 0xB1, 0xF, 0xF, true);  // quad_perm [1,0,3,2]
    // v_perm_b32: bytes 0-3 of `other`'s register are 0-3, of own 4-7
    return __builtin_amdgcn_perm(own, other, (lane & 1) ? 0x07060302u : 0x01000504u);
}

// Block shape: WM x NWN wavefronts, each owning MI x 2 tiles of 32 x 32 (MI * 32 rows x 64
// columns).  WM = 2, MI = 4: 256-row blocks (256 x 128 with 4 wavefronts, 256 x 256 with 8);
// WM = 1: 128-row (MI = 4) and 64-row (MI = 2) blocks for small M.
// SWIGLU: every 16-column tile of the packed weight holds 8 gate columns, then the 8 matching up
// columns; a wavefront's sub-tile 0 gathers the gate columns of its four tiles and sub-tile 1 the
// up columns; the store writes silu(gate) * up, half as wide
// (crates/kiln-model/src/forward.rs:2771-2819 computes gate, up, silu and the product as
// separate bf16 tensors; here the product is formed from the f32 accumulators and rounded once).
// RS: the row sums of A that the offset removal needs are formed inside the kernel from the A
// tiles in LDS (one extra 128-bit LDS read and ~20 VALU instructions per wavefront and stage)
// instead of by the pre-pass kernel: for the small blocks, whose launches are bound by latency,
// this saves a launch and the global reads of the extension operands.
// The LoRA projection (and the extension operand) computed inside the launch that uses them: the
// first `producers` blocks of the grid run lora_project_block (row tiles, K slices one
// after the other) while the others multiply; a block of the product looks at its row tiles' words
// behind its main loop -- long after they were raised -- and reads both operands with ordinary
// loads (no cache on its die has seen those lines since the launch began).  The words live in
// workspace that is all zero between launches (the region lora_tail.h describes: the tile words
// from word kPrefillFoldTileWord of its first replica on); every block counts itself after its
// look, on the replicated counts, and the last one zeroes words and counts.
// A launch without adapters uses the same words for the row sums alone (a_cat == nullptr): its
// producers run rowsum_producer_block.  A block asks for its words a few groups before its main
// loop ends, with a load that lands in LDS by itself (prefill_fold_peek), and waits for them behind
// the loop only if that look came too early.
struct PrefillFold {
    const uint16_t *a_cat;   // bf16 [r_total, K]
    uint16_t *t;             // bf16 [M, RP], behind it the f32 tiles in which K slices meet
    u32x4 *aext;             // the extension operand the producers write
    float *partial;
    int *counters;           // per row tile, zero on entry and exit (not the product's own counters)
    unsigned *words;         // the zeroed region
    int producers;           // a multiple of 8 (the product's blocks keep their dies): project_tiles * kz rounded up, or fewer (WK = 2)
    int row_tiles;           // of 16 rows, a word each
    int project_tiles, kz, steps_per_slice;  // the projection's row tiles (kFoldProjectRows) and K slices
    int consumers;           // blocks of the product (grid padding included)
    int sum_tiles;           // a_cat == nullptr (no adapters): the producers form the row sums only, this many
                             // 16-row tiles each
    LoraScales ls;
};
constexpr int kPrefillFoldTileWord = 32;
// rows per block of a projection inside the product's launch: lora_project_block, or lora_project_stream in launches of one
// block to a compute unit
template <int WK>
constexpr int kFoldProjectRows = WK == 2 ? kStreamRows : 16;
constexpr int kPrefillFoldMaxTiles = kLoraFoldReplicaWords - kPrefillFoldTileWord;
constexpr int kPrefillFoldSpinLimit = 1 << 20;
// where a wavefront's early look at its words lands: the last KiB of the LDS every instance that takes part has
// (the projection's blocks need kProjectLdsBytes16), behind the A ring and the row sums a block may keep there
constexpr int kProjectLdsBytes16 = (16 + kProjectMaxRank) * kProjectRowBytes + kProjectMaxRank * (int)sizeof(float);
constexpr int kFoldPeekOffset = kProjectLdsBytes16 - 1024;

// The row sums of a launch without adapters, as the work of one of its first blocks: the extension
// operand of 16-row tiles [t0, t1) -- a contiguous piece of A, streamed with 24 loads per thread in
// flight; 16 lanes per (row, group), the order of additions of w4a16_prefill_rowsum_kernel, whose
// launch this saves -- written through to memory, then the tiles' words.
template <int THREADS>
__device__ __forceinline__ void rowsum_producer_block(const uint16_t *__restrict__ A, u32x4 *__restrict__ aext, int M,
                                                      int K, int t0, int t1, unsigned *done) {
    constexpr int U = 24, SLOTS = THREADS / 16;
    const int G = K / kGroupK;
    const int r0 = t0 * 16, r1 = min(t1 * 16, M);
    const int items = (r1 - r0) * G;  // item L: the 256 bytes from byte 256 L of the piece on
    const int tid = threadIdx.x, sub = tid & 15, slot = tid >> 4;
    const u32x4 *src = reinterpret_cast<const u32x4 *>(A + (size_t)r0 * K) + sub;
    for (int base = 0; base < items; base += SLOTS * U) {
        u32x4 v[U];
        float sum[U];
#pragma unroll
        for (int u = 0; u < U; ++u)  // items past the end re-read the last one
            v[u] = async_load_b128(src + (size_t)min(base + u * SLOTS + slot, items - 1) * 16);
        unrolled<0, U>([&](auto uc) {
            constexpr int u = decltype(uc)::value;
            // loads complete in issue order: load u has landed when at most the U - 1 - u later ones are pending
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(U - 1 - u));
            pin(v[u]);
            sum[u] = sum_bf16x8(v[u]);
#pragma unroll
            for (int off = 8; off >= 1; off >>= 1) sum[u] += __shfl_xor(sum[u], off, 16);
        });
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int L = base + u * SLOTS + slot;
            if (sub == 0 && L < items) {
                const int row = L / G, g = L - row * G;
                store_b128_through(aext + (size_t)g * M + r0 + row, extension_operand(sum[u]));
            }
        }
    }
    // every wavefront's stores acknowledged, then the words
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __syncthreads();
    for (int t = t0 + tid; t < t1; t += THREADS) __hip_atomic_store(done + t, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A look at the words of rows [m0, m0 + rows) that nobody waits for: one device-scope load per lane
// straight into LDS (256 bytes per wavefront at lds_addr), asked for a few groups before the main
// loop ends so that the round trip runs under its products; prefill_fold_seen() reads the answer.
// Every lane must see a raised word: lanes beyond the last tile look at the last one.
__device__ __forceinline__ void prefill_fold_peek(const PrefillFold &pf, int m0, int rows, int lane, unsigned lds_addr) {
    const int t0 = m0 >> 4, nt = min((rows + 15) >> 4, pf.row_tiles - t0);
    const unsigned *p = pf.words + kPrefillFoldTileWord + t0 + min(lane, nt - 1);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off sc1" : : "v"(p), "s"(lds_addr) : "memory", "m0");
}
__device__ __forceinline__ bool prefill_fold_seen(const unsigned char *lds_slot, int lane) {
    const unsigned f = *reinterpret_cast<const volatile unsigned *>(lds_slot + lane * 4);
    return __builtin_amdgcn_ballot_w64(f == 0u) == 0;
}

// rows [m0, m0 + rows) of T and of the extension operand are in memory
__device__ __forceinline__ void prefill_fold_wait(const PrefillFold &pf, int m0, int rows, int lane) {
    const int t0 = m0 >> 4, nt = min((rows + 15) >> 4, pf.row_tiles - t0);
    int spins = 0;
    for (; spins < kPrefillFoldSpinLimit; ++spins) {
        unsigned f = 1u;
        if (lane < nt) f = __hip_atomic_load(pf.words + kPrefillFoldTileWord + t0 + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__builtin_amdgcn_ballot_w64(f == 0u) == 0) break;
        __builtin_amdgcn_s_sleep(8);
    }
    if (__builtin_expect(spins == kPrefillFoldSpinLimit, 0))
        report_wait_gave_up(error_word_before_fold_words(pf.words), kGaveUpPrefillFold, lane);
}
// one wavefront of block `consumer`, after its look: count the block; the last one zeroes everything
__device__ __forceinline__ void prefill_fold_done(const PrefillFold &pf, int consumer, int lane) {
    const int replica = consumer % kLoraFoldReplicas;
    const unsigned quota = (unsigned)(pf.consumers - replica + kLoraFoldReplicas - 1) / kLoraFoldReplicas;
    const unsigned replicas = (unsigned)min(pf.consumers, kLoraFoldReplicas);
    unsigned before = 0;
    if (lane == 0)
        before = __hip_atomic_fetch_add(pf.words + replica * kLoraFoldReplicaWords + kLoraFoldCountWord, 1u, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT);
    before = (unsigned)__builtin_amdgcn_readfirstlane((int)before);
    if (before != quota - 1u) return;
    if (lane == 0) before = __hip_atomic_fetch_add(pf.words + kLoraFoldTopWord, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    before = (unsigned)__builtin_amdgcn_readfirstlane((int)before);
    if (before != replicas - 1u) return;
    for (int i = lane; i < pf.row_tiles; i += 64)
        __hip_atomic_store(pf.words + kPrefillFoldTileWord + i, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (lane <= kLoraFoldTopWord)
        for (int r = 0; r < kLoraFoldReplicas; ++r)
            __hip_atomic_store(pf.words + r * kLoraFoldReplicaWords + lane, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// INC: c = -136 * sum(a) of every (row, group) is there, in f32, when the launch begins (the pre-pass kernel, or the
// launch that wrote A), and joins the accumulators at the change of group that begins it: the change's multiplication
// by scale(g) / scale(g+1) becomes a multiply-add, and there is no extension contraction (6 % of the products at any
// K, and 2 us a tile).  What it costs is LDS reads: a lane's accumulators lie in 16 rows of every row tile, whose
// values of c it reads (broadcast) in 16-byte pieces, 16 of them a group beside 32 fragments.  For launches of several
// rounds, or of a block for nearly every unit, whose row sums come from in front anyway; where the launch's own blocks form them (RS, and FOLD's producers
// without INC) they are not there when a block begins.  FOLD and INC together: the producers run the projection onto the
// adapters alone.
//
// WK = 2: a block has twice the wavefronts, and each half of them takes half of the block's groups of K, with a ring of
// its own and the barriers in common; the halves' tiles meet in LDS, and each half goes on with half of the rows (the
// exchange of K slices and the store).  For launches of at most one block per compute unit: with one wavefront per SIMD
// nothing covers what one waits for -- a stage's barrier and LDS reads, and its own instruction stream, five cycles an
// instruction, which in 64-row blocks is longer than the products.  An odd number of groups: the second half begins with
// the first's last group and multiplies what it got there by 0.  The halves' stages are met half by half, through a word
// of LDS: half of the wavefronts wait for one another while the other half computes.  (us, one set of wavefronts -> two:
// 128-row blocks 9216 -> 2560 at 777 rows 59.3 -> 53.4; 64-row blocks 9216 -> 2560 at 640 / 512 / 300 rows 54.8 -> 43.3 /
// 41 -> 36.5 / 33.7 -> 28.4, 4096 -> 2560 at 1100 45.5 -> 35.2, 4096 -> 4096 at 777 46 -> 37, 2560 -> 2560 at 777 30 -> 24,
// 1536 -> 1536 at 1300 25.6 -> 17.0.  The sums of K are two shorter ones: error beyond the bf16 rounding 1.79e-4 -> 1.48e-4 of
// the result's norm at 777 x 9216 -> 2560, 14 to 25 % less in each of eight shapes.)
template <int NWN, int WM, int MI, bool SWIGLU, bool RS, bool FOLD = false, bool INC = false, int WK = 1>
__global__ __launch_bounds__(64 * WM * NWN * WK, (WM == 2 && NWN == 4) ? 1 : 2) void w4a16_prefill_kernel(
    const uint16_t *__restrict__ A, const u32x4 *__restrict__ B, const uint16_t *__restrict__ S,
    uint16_t *__restrict__ C, const u32x4 *__restrict__ aext, int M, int N, int K, int Gs, int m_blocks,
    const uint16_t *__restrict__ lora_t, const uint16_t *__restrict__ lora_b, int r_total, int RP, int nb_full,
    int KS, int GSb, float *partial, int *counters, int die_rows, u32x4 *next_aext, bool next_plain, PrefillFold pf) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];  // the A ring; reused by the store
    static_assert(!FOLD || WM * NWN == 4, "the projection's blocks have four wavefronts");
    static_assert(!INC || (!RS && WM == 1 && MI == 4), "the row sums come from in front");
    static_assert(WK == 1 || (WK == 2 && WM == 1), "halves of K: one row of wavefronts");
    if constexpr (FOLD) {
        if ((int)blockIdx.x < pf.producers) {
            const int unit = blockIdx.x;
            if (pf.a_cat == nullptr) {
                const int t0 = unit * pf.sum_tiles;
                if (t0 < pf.row_tiles)
                    rowsum_producer_block<64 * WM * NWN * WK>(A, pf.aext, M, K, t0, min(t0 + pf.sum_tiles, pf.row_tiles),
                                          pf.words + kPrefillFoldTileWord);
                return;
            }
            unsigned *const words = pf.words + kPrefillFoldTileWord;
            if constexpr (WK == 2) {  // in turns, where there are more shares than blocks
                for (int share = unit; share < pf.project_tiles * pf.kz; share += pf.producers) {
                    if (share != unit) __syncthreads();
                    lora_project_stream(lds, A, pf.a_cat, pf.t, M, K, r_total, RP, pf.steps_per_slice, pf.ls, pf.partial, pf.counters,
                                        pf.aext, share % pf.project_tiles, share / pf.project_tiles, pf.kz, words);
                }
            } else if (unit < pf.project_tiles * pf.kz) {
                lora_project_block<16>(lds, A, pf.a_cat, pf.t, M, K, r_total, RP, pf.steps_per_slice, pf.ls, pf.partial, pf.counters,
                                       pf.aext, unit % pf.project_tiles, unit / pf.project_tiles, pf.kz, words);
            }
            return;
        }
    }
    constexpr int BM = WM * MI * 32, BN = 64 * NWN;  // block rows and columns
    constexpr int NW = WM * NWN, NT = 64 * NW * WK;  // wavefronts (of a half of K), threads
    constexpr int kAStageBytes = BM * 32 * 2;        // BM rows x 32 columns of bf16 per stage
    constexpr int APW = (BM / 16) / NW;              // A loads (16 rows each) per wavefront and stage
    static_assert(APW * NW * 16 == BM, "A stage must divide evenly over the wavefronts");
    constexpr int RPW = BM / NW;                     // RS: rows of A each wavefront sums
    static_assert(!RS || RPW % 16 == 0, "row sums are taken 16 rows per read");

    KILN_TL(0);
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = WK == 1 ? 0 : wave_all / NW, wave = WK == 1 ? wave_all : wave_all % NW;  // ... among its half's
    const int wm = wave / NWN, wn = wave % NWN;
    const int G = K / kGroupK;
    const int l32 = lane & 31, h = lane >> 5;

    // Work list.  The first nb_full column blocks are whole tiles (all of K in
    // one block); the remaining column blocks are cut into KS slices of K each,
    // so that a last, partly filled round of tiles still spreads over the whole
    // chip.  Blocks are dispatched in id order: whole tiles first, slices last.
    // Consecutive ids go to different dies.  The 8 dies form a die_rows x
    // (8 / die_rows) grid over (row blocks x units), a unit being a column block
    // or a K slice of one; inside its rectangle a die walks unit by unit, all its
    // row blocks of one unit back to back.  Blocks resident on a die at one time
    // therefore share the few row blocks of A the die owns (they stay in its L2,
    // where the loads that feed the matrix cores three stages ahead must hit) and
    // read each unit's weights from memory once.  (die_rows == 0: no rectangles, prefill_die_rows.)
    int id = blockIdx.x;
    if constexpr (FOLD) id -= pf.producers;
    [[maybe_unused]] const int consumer = id;
    const int n_blocks = N / BN;
    bool sliced, padding;
    int unit, mb;
    if (die_rows == 0) {  // whole tiles one after the other, the same number to every die but for the last
        const int per_die = (m_blocks * n_blocks + 7) >> 3, seq = id >> 3, tile = (id & 7) * per_die + seq;
        unit = tile / m_blocks;
        mb = tile - unit * m_blocks;
        sliced = nb_full == 0;
        padding = seq >= per_die || unit >= n_blocks;
    } else {
        const int die_cols = 8 / die_rows, rows_per_die = (m_blocks + die_rows - 1) / die_rows;
        const int per_die_full = rows_per_die * ((nb_full + die_cols - 1) / die_cols);
        sliced = id >= 8 * per_die_full;
        if (sliced) id -= 8 * per_die_full;
        const int units = sliced ? (n_blocks - nb_full) * KS : nb_full;  // per row block
        const int units_per_die = (units + die_cols - 1) / die_cols;
        const int die = id & 7, seq = id >> 3;
        unit = (die / die_rows) * units_per_die + seq / rows_per_die;
        mb = (die % die_rows) * rows_per_die + seq % rows_per_die;
        padding = seq >= rows_per_die * units_per_die || unit >= units || mb >= m_blocks;
    }
    if (padding) {  // (whole block, before any barrier)
        if constexpr (FOLD) {
            if (wave_all == 0) prefill_fold_done(pf, consumer, lane);  // counted like the others: it will never look
        }
        return;
    }
    int nb = unit, ks = 0;
    if (sliced) {
        nb = nb_full + unit / KS;
        ks = unit % KS;
    }
    const int m0 = mb * BM, n0 = nb * BN;
    // K slice of this block: groups [g_begin, g_end).  With KS > 1 the slices of
    // a tile are combined through the workspace at the end.
    int g_begin = sliced ? ks * GSb : 0, g_end = sliced ? min(G, g_begin + GSb) : G;
    [[maybe_unused]] bool phantom = false;  // the first group is the other half's: its products are dropped
    if constexpr (WK == 2) {
        const int both = g_end - g_begin, each = (both + 1) >> 1;
        phantom = half == 1 && 2 * each != both;
        if (half == 0) g_end = g_begin + each;
        else g_begin = g_end - each;
    }
    // LDS: the halves' rings, then (with the look at a folded launch's words in front) what lies behind a ring
    const int ring = WK == 1 ? 0 : half * (kAStages * kAStageBytes);
    constexpr int kBehindRings = WK * kAStages * kAStageBytes + (WK == 2 && FOLD ? 1024 : 0);
    [[maybe_unused]] constexpr int kPeekAt = WK == 1 ? kFoldPeekOffset : WK * kAStages * kAStageBytes + (INC ? WK * 2 * NW * 256 : 0);

    __shared__ uint32_t s_meeting[2];
    if constexpr (WK == 2) {
        if (tid < 2) s_meeting[tid] = 0;
        wait_lds_reads();  // zero before the barrier in front of the main loop
    }

    // --- A: global -> LDS without passing through registers --------------------
    // A stage is BM rows x 32 columns of bf16 = 64 B per row, 4 units of 16 B; four stages form a ring.
    // Unit c of row r is stored at unit position c ^ ((r >> 2) & 3): with four units
    // per row, any 16 consecutive rows read at one unit index then touch the 16
    // different 16-byte positions of a 256-byte bank line, so the 128-bit fragment
    // reads are bank-conflict free (with (r >> 1) & 3 rows r and r + 8 collided: four
    // conflict cycles on every fragment read, 13 % of the launch's cycles).  One direct
    // load moves 1 KiB = 16 rows: lane i writes LDS slot i, so it fetches row i / 4,
    // unit (i % 4) ^ ((i / 16) & 3).
    // Wavefront w moves the 16-row blocks w, w + NW, ...
    // Rows past M re-read row M - 1: their products are never stored.
    // Addresses are a uniform base in scalar registers, advanced there, plus a lane's constant byte offset.
    uint32_t a_off_g[APW];
#pragma unroll
    for (int p = 0; p < APW; ++p) {
        const int row = min(m0 + (wave + NW * p) * 16 + (lane >> 2), M - 1) - m0;
        a_off_g[p] = (uint32_t)row * (uint32_t)K * 2u + (((lane & 3) ^ ((lane >> 4) & 3)) * 16);
    }
    // WK = 2: where a half's wavefronts meet once a stage (meeting_signal), and how many arrivals there will have been
    [[maybe_unused]] const unsigned meeting = (unsigned)(size_t)(lds_ptr_t)&s_meeting[half];
    [[maybe_unused]] int met = 0;
    [[maybe_unused]] const char *const gave_up_at = uniform(reinterpret_cast<const char *>(counters) + kWsErrorOffset - kGaveUpPrefillMeeting);
    const char *a_ptr = uniform(reinterpret_cast<const char *>(A) + ((size_t)m0 * K + (size_t)g_begin * kGroupK) * 2);  // this group's stages
    const unsigned lds_base = (unsigned)(size_t)(lds_ptr_t)lds, ring_base = lds_base + ring;
    auto load_a = [&](const char *base, int slot) {
#pragma unroll
        for (int p = 0; p < APW; ++p) load_to_lds_b128(base, a_off_g[p], ring_base + slot * kAStageBytes + (wave + NW * p) * 1024);
    };

    // --- B: column sub-tile ni (32 columns = chunks 2ni, 2ni+1 of this wavefront);
    // load v (0/1) fetches lane (l32 % 16) + 16 * (2v + h) of chunk (l32 / 16).
    const int nt_base = (n0 + wn * 64) / kTileN;  // first 16-column tile of this wavefront
    uint32_t b_off[2], s_off[2];
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) {
        // SWIGLU: every 16-column tile holds 8 gate columns, then the 8 matching up columns; sub-tile 0
        // gathers the gate columns of the wavefront's four tiles, sub-tile 1 their up columns, so a lane
        // holds a gate value and its up value in the same register of the two accumulators
        const int nt = SWIGLU ? (l32 >> 3) : 2 * ni + (l32 >> 4);
        const int c = SWIGLU ? (l32 & 7) + 8 * ni : (l32 & 15);
        b_off[ni] = ((uint32_t)nt * (uint32_t)G * 64u + c + 16 * h) * 16u;  // + 512 for v = 1
        s_off[ni] = ((uint32_t)nt * (uint32_t)Gs * kTileN + c) * 2u;
    }
    const int gs_mask = (Gs == 1) ? 0 : -1;
    const int s_step = (Gs == 1) ? 0 : kTileN * 2;  // bytes from a group's scales to the next one's
    const char *b_ptr = uniform(reinterpret_cast<const char *>(B) + ((size_t)nt_base * G + g_begin) * 1024);
    const char *s_ptr = uniform(reinterpret_cast<const char *>(S) + (size_t)nt_base * Gs * kTileN * 2 + (size_t)(g_begin & gs_mask) * kTileN * 2);
    // a zero scale would break the running rescale below; it is replaced by a
    // value too small to matter (the same value in the extension contraction)
    auto scale_value = [&](uint32_t raw) {
        const float sv = f16_bits_to_f32((uint16_t)raw);
        return sv == 0.f ? 0x1p-40f : sv;
    };

    const DequantConsts dq = dequant_consts();
    // fragment read offsets inside a stage for the two k16 steps of a stage:
    // row (wm*MI*32 + mi*32 + l32), unit (2*step + h) ^ ((row >> 2) & 3)
    int a_off[2];
#pragma unroll
    for (int sp = 0; sp < 2; ++sp)
        a_off[sp] = ring + (wm * MI * 32 + l32) * 64 + (((2 * sp + h) ^ ((l32 >> 2) & 3)) * 16);

    f32x16 acc[MI][2];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < 2; ++ni)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mi][ni][r] = 0.f;

    // --- the main loop's schedule ---------------------------------------------
    // The matrix cores bound this loop, so everything else is placed under their products, by hand: a stage
    // (32 of K) is MI phases of four products each, phase mi = row tile mi, both column sub-tiles, both k16 steps.
    //   * Fragments of A are read a stage ahead: the two of row tile mi right behind phase mi's products, for the
    //     next stage.  They are used MI phases later, so no product waits for LDS.
    //   * Behind phase 0 comes the stage's one barrier: the next stage has landed (counted waits), and every
    //     wavefront holds all of this stage's fragments, so its slot is free at once -- the loads asked for then
    //     fill it, four stages ahead of their use with a ring of four.
    //   * The next stage's four operands of B are expanded from their words half an operand at a time (3 or 4
    //     vector instructions) behind a product each.
    //   * The group's change of scale (below) goes tile by tile behind products of other tiles: from phase 1 of
    //     the group's last stage on, and over the first phases of the next group's first stage.
    // sched_barrier pins the order; left to itself the compiler gathers the fragment reads, the expansions and the
    // 128 multiplies of a group in front of the products that need them, and the matrix cores idle there (measured
    // with such a loop, 2560 -> 2 x 9216 at 8192 rows: 56 % of the cycles busy).
    u32x4 bw[2][2], bw_next[2][2];  // the group's words of B, and the next group's
    uint32_t sc_raw[2];
    auto request_b = [&](u32x4(&w)[2][2], const char *base, const char *sbase) {
#pragma unroll
        for (int ni = 0; ni < 2; ++ni) {
            asm volatile("global_load_dwordx4 %0, %1, %2" : "=&v"(w[ni][0]) : "v"(b_off[ni]), "s"(base) : "memory");
            asm volatile("global_load_dwordx4 %0, %1, %2 offset:512" : "=&v"(w[ni][1]) : "v"(b_off[ni]), "s"(base) : "memory");
            load_u16(sc_raw[ni], sbase, s_off[ni]);
        }
    };
    // prologue: the first group's words, four stages of A
    // INC: c of a group's rows, [row] f32, in two slots that take turns; every wavefront asks for 64 rows of it
    // (wavefronts beyond the block's rows for a copy nobody reads, so that all count the same loads)
    constexpr int kSumSlot = NW * 256;
    static_assert((kAStages * kAStageBytes) % (2 * kSumSlot) == 0, "slots alternate by one bit of their offset");
    const int c_slots = WK * kAStages * kAStageBytes + (WK == 1 ? 0 : half * (2 * kSumSlot));
    [[maybe_unused]] int c_at = c_slots + h * 16;                  // this group's slot; the next one's is c_at ^ kSumSlot
    [[maybe_unused]] const char *c_ptr = nullptr;                  // this group's c in memory
    [[maybe_unused]] const uint32_t c_off = (uint32_t)min(m0 + (wave % (BM / 64)) * 64 + lane, M - 1) * 4u;
    [[maybe_unused]] int c_to = c_slots + wave * 256;              // offsets: the slots' bit is theirs, not the base's
    if constexpr (INC) c_ptr = uniform(reinterpret_cast<const char *>(aext) + (size_t)g_begin * M * 4);
    request_b(bw, b_ptr, s_ptr);
    if constexpr (INC) load_to_lds_b32(c_ptr, c_off, lds_base + c_to);
#pragma unroll
    for (int st = 0; st < 4; ++st) load_a(a_ptr + st * 64, st);
    wait_vector_loads<3 * APW>();  // the words and stage 0
    __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
    float sc[2], f[2] = {1.f, 1.f};
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) {
        pin(bw[ni][0]);
        pin(bw[ni][1]);
        pin(sc_raw[ni]);
        sc[ni] = WK == 2 && phantom ? 0.f : scale_value(sc_raw[ni]);  // (the change to the next group's multiplies by it)
    }
    bf16x8 af[MI][2], bf[2][2];
    auto read_a = [&](auto slotc, int mi) {
#pragma unroll
        for (int sp = 0; sp < 2; ++sp)
            af[mi][sp] = *reinterpret_cast<const bf16x8 *>(lds + decltype(slotc)::value * kAStageBytes + a_off[sp] + mi * 32 * 64);
    };
    // RS: c[group][row] = -136 * (row sum of the group), f32, behind the ring.  Wavefront w sums rows w * RPW ...: lane ->
    // row lane / 4, unit lane % 4 of a stage; the four lanes of a row meet when the group ends.
    int g_now = g_begin;
    [[maybe_unused]] float gsum[RS ? RPW / 16 : 1] = {};
    [[maybe_unused]] float *csum = reinterpret_cast<float *>(lds + kBehindRings) + half * (g_end - g_begin) * BM;
    [[maybe_unused]] auto sum_rows = [&](auto slotc) {
#pragma unroll
        for (int rr = 0; rr < RPW / 16; ++rr) {
            const int row = wave * RPW + rr * 16 + (lane >> 2);
            const u32x4 v = *reinterpret_cast<const u32x4 *>(lds + ring + decltype(slotc)::value * kAStageBytes + row * 64 + (((lane & 3) ^ ((row >> 2) & 3)) * 16));
            gsum[rr] += sum_bf16x8(v);
        }
    };
    [[maybe_unused]] auto flush_rows = [&](int gl) {
#pragma unroll
        for (int rr = 0; rr < RPW / 16; ++rr) {
            float s8 = gsum[rr];
            s8 += dpp_move<0xB1>(s8);  // quad_perm [1,0,3,2]
            s8 += dpp_move<0x4E>(s8);  // quad_perm [2,3,0,1]
            csum[gl * BM + wave * RPW + rr * 16 + (lane >> 2)] = -kCodeBias * s8;  // the same value from all four lanes
            gsum[rr] = 0.f;
        }
    };
    auto word_of = [](const u32x4(&w)[2][2], auto qc, int ni, int sp) {
        constexpr int q = decltype(qc)::value;
        return (q == 0) ? w[ni][sp].x : (q == 1) ? w[ni][sp].y : (q == 2) ? w[ni][sp].z : w[ni][sp].w;
    };
    if constexpr (RS) sum_rows(std::integral_constant<int, 0>{});
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) read_a(std::integral_constant<int, 0>{}, mi);
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
        for (int sp = 0; sp < 2; ++sp) bf[ni][sp] = codes_to_bf16x8(word_of(bw, std::integral_constant<int, 0>{}, ni, sp), dq);

    // The operands of the extension contraction (behind the main loop) ride in the ring like further stages: an
    // extension stage is four groups, [group][row] 16 bytes of the rows' sums (not with RS, whose sums are in LDS),
    // and beside it the four groups' scales of every wavefront's 64 columns, [group][column] fp16.  The last group
    // of the main loop asks for the first four in place of further stages of A.
    const int ng = g_end - g_begin;
    const char *const s_base = s_ptr;
    constexpr int kExtLoads = INC ? 0 : (RS ? 0 : APW) + 2;  // per wavefront and extension stage
    const uint32_t ext_off = (uint32_t)min(m0 + (RS ? 0 : (wave % (BM / 64)) * 64) + lane, M - 1) * 16u;
    auto ext_scales = [&](int slot) {
        return RS ? ring + slot * kAStageBytes + wave * 512 : kBehindRings + ((half * kAStages + slot) * NW + wave) * 512;
    };
    auto request_ext = [&](int e, int slot) {  // groups past the last re-read it
        if constexpr (!RS) {
#pragma unroll
            for (int p = 0; p < APW; ++p) {
                const int i = wave + NW * p, g = g_begin + min(4 * e + i / (BM / 64), ng - 1);
                load_to_lds_b128(uniform(reinterpret_cast<const char *>(aext + (size_t)g * M)), ext_off,
                                 ring_base + slot * kAStageBytes + i * 1024);
            }
        }
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            const int g = min(4 * e + 2 * v + h, ng - 1) & gs_mask;
            const uint32_t off = ((uint32_t)((lane >> 3) & 3) * (uint32_t)Gs + (uint32_t)g) * (kTileN * 2) + (lane & 7) * 4;
            load_to_lds_b32(s_base, off, lds_base + ext_scales(slot) + v * 256);
        }
    };
    // INC: the change of group in work items of four registers -- (row tile, quarter, column sub-tile) -- behind the
    // products kChangeAt ... of the old group's last stage (row tiles of the first half) and of the new group's first
    // (the others, counted without the four products in front of the barrier), kChangeRoom of them, a quarter's c read
    // kChangeLead products before its first use.
    constexpr int kChangeAt = 2, kChangeRoom = 10, kChangeLead = 2;
    static_assert(kChangeLead <= kChangeAt, "the next group's c is read behind the barrier that shows it");
    if constexpr (INC) {
#pragma unroll
        for (int mi = 0; mi < MI / 2; ++mi)  // the others begin at 0 and take c in the first stage
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f32x4 c = *reinterpret_cast<const f32x4 *>(lds + c_at + mi * 128 + i * 32);
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[mi][0][4 * i + r] = acc[mi][1][4 * i + r] = c[r];
            }
    }
    // one group; LAST: no further group; PEEK: ask for the words of a folded launch
    auto group = [&](auto lastc, auto peekc) {
        constexpr bool LAST = decltype(lastc)::value, PEEK = decltype(peekc)::value;
        unrolled<0, 4>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            constexpr bool ahead = !(LAST && q == 3);  // there is a next stage
            u32x4 bn[2][2];
            [[maybe_unused]] f32x4 cq[INC ? MI * 2 : 1];
            // Loads complete in issue order; behind the next stage's there are those of the two stages after
            // it (in the last group extension stages take the place of stages) and, unless they are needed now,
            // the next group's six, its c and the look at the words.
            constexpr int a_behind = LAST && q > 0 ? (q == 1 ? 1 : 0) : 2;
            constexpr int others = (!LAST && (q == 1 || q == 2)) ? 6 + (PEEK ? 1 : 0) + (INC ? 1 : 0) : 0;
            constexpr int kStageLanded = a_behind * APW + (2 - a_behind) * kExtLoads + others;
            if constexpr (WK == 2) {  // the half's wavefronts meet: this one's part of the next stage is there, its reads of this stage asked for
                wait_vector_loads<kStageLanded>();
                meeting_signal(meeting);
                met += NW;
            }
            [[maybe_unused]] uint32_t seen_met = 0;
            unrolled<0, MI>([&](auto mc) {
                constexpr int mi = decltype(mc)::value;
                unrolled<0, 4>([&](auto jc) {
                    constexpr int j = decltype(jc)::value, ni = j & 1, sp = j >> 1, slot = 4 * mi + j;
                    if constexpr (WK == 2 && slot == 3) meeting_look(meeting, seen_met);
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[mi][sp], bf[ni][sp], acc[mi][ni], 0, 0, 0);
                    // behind this product: halves of the next stage's operands of B ...
                    constexpr int first = q == 3 ? 4 : 0, room = 4 * MI - first;  // (the next group's words are there behind the barrier)
                    if constexpr (ahead && slot >= first) {
                        constexpr int h0 = (slot - first) * 8 / room, h1 = (slot - first + 1) * 8 / room;
                        unrolled<h0, h1>([&](auto hc) {
                            constexpr int hh = decltype(hc)::value, en = (hh >> 1) & 1, es = hh >> 2;
                            const uint32_t w = q == 3 ? word_of(bw_next, std::integral_constant<int, 0>{}, en, es)
                                                      : word_of(bw, std::integral_constant<int, (q + 1) & 3>{}, en, es);
                            if constexpr ((hh & 1) == 0) {
                                bn[en][es].x = (w & dq.mask) | dq.magic;
                                bn[en][es].y = ((w >> 4) & dq.mask) | dq.magic;
                            } else {
                                bn[en][es].z = ((w >> 8) & dq.mask) | dq.magic;
                                bn[en][es].w = ((w >> 12) & dq.mask) | dq.magic;
                            }
                        });
                    }
                    // ... and a part of the change of scale
                    // tile t is complete behind phase t / 2 of the last stage and needed by that phase of the next
                    // stage; MI = 4: tiles 0 | 1 2 | 3 4 in phases 1, 2, 3, tiles 5 | 6 | 7 in phases 0, 1, 2 of the next group
                    constexpr int t0 = q == 3 ? (MI == 4 ? (mi < 2 ? 0 : 2 * mi - 3) : 0) : (MI == 4 ? 5 + mi : 2);
                    constexpr int t1 = q == 3 ? (MI == 4 ? (mi == 0 ? 0 : 2 * mi - 1) : (mi == 0 ? 0 : 2)) : (MI == 4 ? 6 + mi : (mi == 0 ? 4 : 2));
                    if constexpr (INC && ((q == 3 && !LAST) || q == 0)) {
                        constexpr int at = slot - (q == 3 ? 4 : 0) - kChangeAt, items = MI * 4;
                        constexpr int rt0 = q == 3 ? 0 : MI / 2;
                        constexpr auto begin_of = [](int p) { return p < 0 ? 0 : p > kChangeRoom ? items : p * items / kChangeRoom; };
                        unrolled<begin_of(at + kChangeLead), begin_of(at + kChangeLead + 1)>([&](auto ec) {
                            constexpr int e = decltype(ec)::value, quarter = e >> 1;
                            if constexpr ((e & 1) == 0)
                                cq[quarter] = *reinterpret_cast<const f32x4 *>(lds + (q == 3 ? c_at ^ kSumSlot : c_at) +
                                                                               (rt0 + (quarter >> 2)) * 128 + (quarter & 3) * 32);
                        });
                        unrolled<begin_of(at), begin_of(at + 1)>([&](auto ec) {
                            constexpr int e = decltype(ec)::value, quarter = e >> 1, en = e & 1;
                            f32x16 &a = acc[rt0 + (quarter >> 2)][en];
#pragma unroll
                            for (int r = 0; r < 4; ++r) a[4 * (quarter & 3) + r] = fmaf(a[4 * (quarter & 3) + r], f[en], cq[quarter][r]);
                            // c outlives its last use: left to itself the compiler lets that one write over c's registers
                            // and copies the accumulator tile together again, or spills
                            if constexpr (en == 1) asm volatile("" : : "v"(cq[quarter]));
                        });
                    }
                    if constexpr (!INC && ((q == 3 && !LAST) || (q == 0 && mi < MI - 1))) {
                        unrolled<t0, t1>([&](auto tc) {
                            constexpr int t = decltype(tc)::value;
#pragma unroll
                            for (int r = 4 * j; r < 4 * j + 4; ++r) acc[t >> 1][t & 1][r] *= f[t & 1];
                        });
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
                if constexpr (mi == 0) {
                    if constexpr (WK == 2) {
                        meeting_wait(meeting, seen_met, met, gave_up_at);
                    } else {
                        wait_vector_loads<kStageLanded>();
                        wait_lds_reads();
                        __builtin_amdgcn_s_barrier();
                    }
                    asm volatile("" : : : "memory");
                    if constexpr (!LAST) {
                        load_a(a_ptr + (q + 4) * 64, q);
                        if constexpr (q == 0 && !INC) request_b(bw_next, b_ptr + 1024, s_ptr + s_step);
                        if constexpr (q == 3) {
#pragma unroll
                            for (int i = 0; i < 2; ++i) {
                                pin(bw_next[i][0]);
                                pin(bw_next[i][1]);
                                pin(sc_raw[i]);
                                // Running rescale: the accumulator holds (sum so far) / scale(g).  Switching to
                                // the next group's scale multiplies it by scale(g) / scale(g+1); after the last
                                // group, by scale(g).  Nothing is ever rounded to bf16.
                                const float sn = scale_value(sc_raw[i]);
                                f[i] = sc[i] * __builtin_amdgcn_rcpf(sn);
                                sc[i] = sn;
                            }
                        }
                    }
                    if constexpr (LAST && !INC) request_ext(q, q);
                    if constexpr (PEEK && q == 0) prefill_fold_peek(pf, m0, min(BM, M - m0), lane, lds_base + kPeekAt + wave * 256);
                }
                if constexpr (INC && q == 0 && mi == MI - 1 && !LAST) {
                    // three phases later than without INC: the registers are c's until then
                    request_b(bw_next, b_ptr + 1024, s_ptr + s_step);
                    load_to_lds_b32(c_ptr + (size_t)M * 4, c_off, lds_base + (c_to ^ kSumSlot));
                }
                if constexpr (ahead) {
                    if constexpr (RS && mi == 0) {
                        if constexpr (q == 3) flush_rows(g_now - g_begin);
                        sum_rows(std::integral_constant<int, (q + 1) & 3>{});
                    }
                    read_a(std::integral_constant<int, (q + 1) & 3>{}, mi);
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
            if constexpr (ahead) {
#pragma unroll
                for (int ni = 0; ni < 2; ++ni)
#pragma unroll
                    for (int sp = 0; sp < 2; ++sp) bf[ni][sp] = __builtin_bit_cast(bf16x8, bn[ni][sp]);
            }
        });
    };
    auto next_group = [&]() {
#pragma unroll
        for (int ni = 0; ni < 2; ++ni)
#pragma unroll
            for (int v = 0; v < 2; ++v) bw[ni][v] = bw_next[ni][v];
        a_ptr += 256;
        b_ptr += 1024;
        s_ptr += s_step;
        if constexpr (INC) {
            c_ptr += (size_t)M * 4;
            c_at ^= kSumSlot;
            c_to ^= kSumSlot;
        }
        ++g_now;
    };
    while (g_now + 1 + (FOLD ? 1 : 0) < g_end) {
        group(std::false_type{}, std::false_type{});
        next_group();
    }
    if constexpr (FOLD) {
        // The rows of this block in the extension operand and in T are written during this launch.  The look at
        // their words is asked for two groups before the main loop ends and answered one group later; the
        // operands may be asked for from then on.
        bool seen = false;
        if (ng > 1) {
            group(std::false_type{}, std::true_type{});
            next_group();
            seen = prefill_fold_seen(lds + kPeekAt + wave * 256, lane);  // (WK = 2: of either half's wavefront; raised is raised)
        }
        if (!seen) prefill_fold_wait(pf, m0, min(BM, M - m0), lane);
    }
    group(std::true_type{}, std::false_type{});
    if constexpr (RS) {
        flush_rows(g_now - g_begin);
        __syncthreads();  // every wavefront's row sums are in LDS
    }
    f[0] = sc[0];
    f[1] = sc[1];
#pragma unroll
    for (int t = 0; t < 2 * MI; ++t) {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t >> 1][t & 1][r] *= f[t & 1];
    }

    KILN_TL(1);
    // --- remove the 136 * sum(a) * scale surplus: extension contraction ------
    // A product step covers two groups (lanes 0-31 and 32-63), 8 slots each; an extension stage is two steps.
    // While one step is multiplied the other's operands are read from LDS: a stage's second step behind its first
    // one's products, the next stage's first step behind the barrier between the two steps -- there the next
    // stage has landed, and every wavefront holds what it needs of this one, whose slot takes the fourth ahead.
    struct ExtStep {
        bf16x8 a[RS ? 1 : MI];
        float c[RS ? MI : 1];
        uint32_t s[2];
    };
    auto ext_read = [&](int e, int u, ExtStep &x) {
        const int slot = e & 3;
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
            const int row = wm * MI * 32 + mi * 32 + l32;
            if constexpr (RS) x.c[mi] = csum[min(4 * e + 2 * u + h, ng - 1) * BM + row];
            else x.a[mi] = *reinterpret_cast<const bf16x8 *>(lds + ring + slot * kAStageBytes + ((2 * u + h) * BM + row) * 16);
        }
#pragma unroll
        for (int ni = 0; ni < 2; ++ni) {
            const int col = SWIGLU ? (l32 >> 3) * 16 + (l32 & 7) + 8 * ni : 32 * ni + l32;
            x.s[ni] = *reinterpret_cast<const uint16_t *>(lds + ext_scales(slot) + (2 * u + h) * 128 + col * 2);
        }
    };
    auto ext_multiply = [&](int e, int u, const ExtStep &x) {
        const bool live = 4 * e + 2 * u + h < ng && (WK == 1 || !phantom || 4 * e + 2 * u + h > 0);
        bf16x8 bx[2];
#pragma unroll
        for (int ni = 0; ni < 2; ++ni) {
            const float sv = scale_value(x.s[ni]);
            const uint32_t hi = __builtin_bit_cast(uint32_t, sv) & 0xFFFF0000u;
            const float lo_f = sv - __builtin_bit_cast(float, hi);  // exact: f16 has 11 significant bits
            const uint32_t pair = live ? ((hi >> 16) | (__builtin_bit_cast(uint32_t, lo_f) & 0xFFFF0000u)) : 0u;
            bx[ni] = __builtin_bit_cast(bf16x8, u32x4{pair, pair, pair, 0u});
        }
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
            bf16x8 ax;
            if constexpr (RS) {
                // c split exactly into three bf16 terms: [hi, hi, mid, mid, lo, lo, 0, 0]
                const float c = x.c[mi];
                const uint32_t hi = __builtin_bit_cast(uint32_t, c) & 0xFFFF0000u;
                const float r1 = c - __builtin_bit_cast(float, hi);                     // exact
                const uint32_t mid = __builtin_bit_cast(uint32_t, r1) & 0xFFFF0000u;
                const float r2 = r1 - __builtin_bit_cast(float, mid);                   // exact, <= 8 significant bits
                const uint32_t lo = __builtin_bit_cast(uint32_t, r2) & 0xFFFF0000u;
                ax = __builtin_bit_cast(bf16x8, live ? u32x4{(hi >> 16) | hi, (mid >> 16) | mid, (lo >> 16) | lo, 0u} : u32x4{0u, 0u, 0u, 0u});
            } else {
                ax = x.a[mi];
            }
#pragma unroll
            for (int ni = 0; ni < 2; ++ni) acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ax, bx[ni], acc[mi][ni], 0, 0, 0);
        }
    };
    if constexpr (!INC) {
        ExtStep x0, x1;
        ext_read(0, 0, x0);  // visible since the last group's last barrier
        for (int e = 0; 4 * e < ng; ++e) {
            ext_read(e, 1, x1);
            __builtin_amdgcn_sched_barrier(0);
            ext_multiply(e, 0, x0);
            __builtin_amdgcn_sched_barrier(0);
            if (4 * (e + 1) < ng) {
                // behind the next stage there are those of the two stages after it, where they were asked for
                if (e == 0 || 4 * (e + 3) < ng) wait_vector_loads<2 * kExtLoads>();
                else wait_vector_loads<0>();
                wait_lds_reads();
                __builtin_amdgcn_s_barrier();
                asm volatile("" : : : "memory");
                if (4 * (e + 4) < ng) request_ext(e + 4, e & 3);
                ext_read(e + 1, 0, x0);
            }
            __builtin_amdgcn_sched_barrier(0);
            ext_multiply(e, 1, x1);
        }
    }
    wait_vector_loads<0>();  // stages asked for past the end still write to LDS, which the store reuses behind its barrier
    // (Every wavefront has looked at the words: the barriers of the last group's stages are behind that.  Halves of K have
    // none in common there: their block is counted behind the barrier in front of their meeting.)
    if constexpr (FOLD && WK == 1) {
        if (wave_all == 0) prefill_fold_done(pf, consumer, lane);
    }

    // --- fused LoRA epilogue: y += T * B_cat^T with T = scaled x * A_cat^T from the
    // pre-pass (crates/kiln-model/src/lora_loader.rs:213-232, unfused at the call
    // sites forward.rs:2932-2939).  RP / 16 more k16 steps on the same accumulators.
    for (int u = 0; u < (ks == 0 && half == 0 ? RP / 16 : 0); ++u) {  // the LoRA term belongs to one slice (and half) only
        const int j8 = 16 * u + 8 * h;  // this lane's 8 rank columns
        bf16x8 lb[2];
#pragma unroll
        for (int ni = 0; ni < 2; ++ni) {
            // the lane's column of accumulator ni, as the main loop maps it (SWIGLU: gate columns of four
            // tiles in accumulator 0, their up columns in 1; lora_b's rows are in the packed column order)
            const int bcol = SWIGLU ? 16 * (l32 >> 3) + 8 * ni + (l32 & 7) : ni * 32 + l32;
            const uint16_t *bp = lora_b + (size_t)(n0 + wn * 64 + bcol) * r_total + j8;
            if ((r_total & 7) == 0 && j8 + 8 <= r_total) {
                lb[ni] = *reinterpret_cast<const bf16x8 *>(bp);
            } else {
                uint16_t tmp[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) tmp[i] = (j8 + i < r_total) ? bp[i] : (uint16_t)0;
                u32x4 r = {tmp[0] | ((uint32_t)tmp[1] << 16), tmp[2] | ((uint32_t)tmp[3] << 16),
                           tmp[4] | ((uint32_t)tmp[5] << 16), tmp[6] | ((uint32_t)tmp[7] << 16)};
                lb[ni] = __builtin_bit_cast(bf16x8, r);
            }
        }
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
            int row = m0 + wm * MI * 32 + mi * 32 + l32;
            row = row < M ? row : M - 1;
            const bf16x8 la = *reinterpret_cast<const bf16x8 *>(lora_t + (size_t)row * RP + j8);
#pragma unroll
            for (int ni = 0; ni < 2; ++ni)
                acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(la, lb[ni], acc[mi][ni], 0, 0, 0);
        }
    }

    // --- the halves of K meet in LDS: a wavefront hands the other half's wavefront of its columns that one's rows and
    // adds what it gets to its own, the earlier groups' sum first (a + b is b + a)
    constexpr int MIS = MI / WK;  // row tiles a wavefront goes on with
    const int row_first = wm * MI * 32 + half * (MIS * 32);
    if constexpr (WK == 2) {
        __syncthreads();  // every wavefront is done with the rings, and has looked at a folded launch's words
        if constexpr (FOLD) {
            if (wave_all == 0) prefill_fold_done(pf, consumer, lane);
        }
        f32x4 *box = reinterpret_cast<f32x4 *>(lds) + lane;  // [half][wavefront][row tile, sub-tile, four registers][lane]
        auto four = [](const f32x16 &a, int i) { return f32x4{a[4 * i], a[4 * i + 1], a[4 * i + 2], a[4 * i + 3]}; };
        auto hand_over = [&](auto firstc) {
            f32x4 *mine = box + (half * NW + wave) * (MIS * 8) * 64;
            unrolled<0, MIS * 8>([&](auto ec) {
                constexpr int e = decltype(ec)::value;
                mine[e * 64] = four(acc[decltype(firstc)::value + e / 8][(e / 4) & 1], e & 3);
            });
        };
        if (half == 0) hand_over(std::integral_constant<int, MIS>{});
        else hand_over(std::integral_constant<int, 0>{});
        __syncthreads();
        const f32x4 *got = box + ((half ^ 1) * NW + wave) * (MIS * 8) * 64;
        auto add = [&](auto firstc) {
            unrolled<0, MIS * 8>([&](auto ec) {
                constexpr int e = decltype(ec)::value;
                const f32x4 g = got[e * 64], own = four(acc[decltype(firstc)::value + e / 8][(e / 4) & 1], e & 3);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[e / 8][(e / 4) & 1][4 * (e & 3) + i] = own[i] + g[i];
            });
        };
        if (half == 0) add(std::integral_constant<int, 0>{});
        else add(std::integral_constant<int, MIS>{});
    }

    // --- store.  Register r of a 32x32 tile holds row 8*(r/4) + 4*h + r%4,
    // column l32: a lane owns one column.  Each wavefront transposes its
    // (MI * 32) x 64 tile through its own piece of LDS (the now idle A ring) as bf16, then
    // writes rows with 128-bit stores: 8 lanes cover the 128 contiguous bytes
    // of one row of the tile.
    KILN_TL(2);
    if (sliced && KS > 1) {
        // Combine the K slices of this tile.  Every block writes its f32 partial
        // tile with device-scope accesses, 16 bytes each (registers 4 i ... 4 i + 3 of tile (mi, ni) of thread t at
        // 16-byte unit ((mi*2+ni)*4 + i) * NT + t: coalesced both ways); the last block to
        // arrive reads all KS partial tiles back and adds them in slice order,
        // so the result does not depend on arrival order.
        __shared__ int s_last;
        const int tile = (nb - nb_full) * m_blocks + mb;
        float *mine = partial + ((size_t)tile * KS + ks) * (BM * BN) + tid * 4;
#pragma unroll
        for (int mi = 0; mi < MIS; ++mi)
#pragma unroll
            for (int ni = 0; ni < 2; ++ni)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const f32x4 v = {acc[mi][ni][4 * i], acc[mi][ni][4 * i + 1], acc[mi][ni][4 * i + 2], acc[mi][ni][4 * i + 3]};
                    store_b128_device_scope(mine + ((mi * 2 + ni) * 4 + i) * NT * 4, __builtin_bit_cast(u32x4, v));
                }
        // each wavefront waits until its own stores have been acknowledged (a barrier alone
        // orders nothing outside the workgroup); after the barrier the arrival is counted
        wait_vector_loads<0>();
        __syncthreads();
        KILN_TL(3);
        if (tid == 0)
            s_last = (__hip_atomic_fetch_add(counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == KS - 1);
        __syncthreads();
        if (!s_last) return;
        // 16 loads (64 registers) a batch at most, a round trip each.  The block's own part is
        // still in its registers: as slice 0 or 1 the others are added to it as they come (a + b is b + a, so the
        // sum is the one in slice order); further on the sum before it would need registers of its own, and
        // it is read back like the others.
        constexpr int kBatch = MIS * 8 < 16 ? MIS * 8 : 16;
        const float *all = partial + (size_t)tile * KS * (BM * BN) + tid * 4;
        for (int s2 = 0; s2 < KS; ++s2) {
            if (ks < 2 && s2 == ks) continue;
            const bool first = ks >= 2 && s2 == 0;
            const float *src = all + (size_t)s2 * (BM * BN);
#pragma unroll
            for (int batch = 0; batch < MIS * 8 / kBatch; ++batch) {
                u32x4 t[kBatch];
#pragma unroll
                for (int i = 0; i < kBatch; ++i) load_b128_device_scope(t[i], src + (batch * kBatch + i) * NT * 4);
                wait_vector_loads<0>();
#pragma unroll
                for (int i = 0; i < kBatch; ++i) {
                    pin_loaded(t[i]);
                    const f32x4 v = __builtin_bit_cast(f32x4, t[i]);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int at = 4 * (i & 3) + r;
                        f32x16 &a = acc[batch * (kBatch / 8) + i / 8][(i / 4) & 1];
                        a[at] = first ? v[r] : a[at] + v[r];
                    }
                }
            }
        }
        if (tid == 0) __hip_atomic_store(counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        KILN_TL(4);
    }
    __syncthreads();  // every wavefront is done reading the A ring
    if constexpr (SWIGLU) {
        // acc[mi][0] holds gate, acc[mi][1] the matching up columns: h = gate / (1 + exp(-gate)) * up.
        // The wavefront's tile becomes (MIS * 32) x 32: rows of 64 bytes, 4 lanes per row.
        uint16_t *tile = reinterpret_cast<uint16_t *>(lds + wave_all * (MIS * 32 * 32 * 2));  // [MIS * 32][32] bf16
        [[maybe_unused]] float *unit_sums = reinterpret_cast<float *>(lds + WK * NW * (MIS * 32 * 32 * 2));  // [BM][16 units of 8 columns]
        uint32_t *dst[2];  // of row pairs 0 and 2 of every four
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int row = 4 * h + 2 * i + (lane & 1);
            dst[i] = reinterpret_cast<uint32_t *>(tile + row * 32 + ((((l32 >> 3) ^ (row & 3)) << 3) | (l32 & 6)));
        }
#pragma unroll
        for (int mi = 0; mi < MIS; ++mi)
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                float hval[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const float gate = acc[mi][0][r + i], up = acc[mi][1][r + i];
                    hval[i] = gate * __builtin_amdgcn_rcpf(1.f + __expf(-gate)) * up;
                }
                dst[(r >> 1) & 1][(mi * 32 + 8 * (r >> 2)) * 16] = neighbours_of_a_row(hval[0], hval[1], lane);
            }
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
#pragma unroll
        for (int p = 0; p < MIS * 2; ++p) {
            const int row = p * 16 + (lane >> 2), unit = lane & 3;
            const u32x4 v = *reinterpret_cast<const u32x4 *>(tile + row * 32 + ((unit ^ (row & 3)) << 3));
            const int grow = m0 + row_first + row;
            if (grow < M)
                *reinterpret_cast<u32x4 *>(C + (size_t)grow * (N / 2) + (n0 + wn * 64) / 2 + unit * 8) = v;
            if constexpr (WM == 1 && NWN == 4) {
                if (next_aext) unit_sums[(row_first + row) * 16 + wn * 4 + unit] = sum_bf16x8(v);
            }
        }
        if constexpr (WM == 1 && NWN == 4) {
            // The rows' sums for a GEMM over this output (an MLP's down projection): the block's 128 output columns are
            // one group of that GEMM's K, so its rows' sums are formed here, from the stored bf16 values and in the pre-pass
            // kernel's order of additions (bit-equal), and no pass over H is needed for them: 16 bytes per 256 of H
            // written here, from values already in registers (2560 -> 2 x 9216 -> 2560: 8192 rows 973 -> 953 us, the pass read
            // 151 MB in a launch of its own; 2048 rows 282 -> 276, blocks of the down projection's own launch read them).
            if (next_aext) {
                __syncthreads();
                if (tid < BM && m0 + tid < M) {
                    float u[16];
#pragma unroll
                    for (int i = 0; i < 4; ++i) *reinterpret_cast<f32x4 *>(u + 4 * i) = *reinterpret_cast<const f32x4 *>(unit_sums + tid * 16 + 4 * i);
#pragma unroll
                    for (int off = 8; off >= 1; off >>= 1)
#pragma unroll
                        for (int i = 0; i < off; ++i) u[i] += u[i + off];
                    store_row_sum(next_aext, (size_t)nb * M + m0 + tid, u[0], next_plain);
                }
            }
        }
    } else {
        uint16_t *tile = reinterpret_cast<uint16_t *>(lds + wave_all * (MIS * 32 * 64 * 2));  // [MIS * 32][64] bf16
        uint32_t *dst[2][2];  // of sub-tile ni, row pairs 0 and 2 of every four
#pragma unroll
        for (int ni = 0; ni < 2; ++ni)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                // 16-byte unit index XOR (row & 7): keeps the row reads below conflict free
                const int row = 4 * h + 2 * i + (lane & 1), col = ni * 32 + l32;
                dst[ni][i] = reinterpret_cast<uint32_t *>(tile + row * 64 + ((((col >> 3) ^ (row & 7)) << 3) | (col & 6)));
            }
#pragma unroll
        for (int mi = 0; mi < MIS; ++mi)
#pragma unroll
            for (int ni = 0; ni < 2; ++ni)
#pragma unroll
                for (int r = 0; r < 16; r += 2)
                    dst[ni][(r >> 1) & 1][(mi * 32 + 8 * (r >> 2)) * 32] = neighbours_of_a_row(acc[mi][ni][r], acc[mi][ni][r + 1], lane);
        // same wavefront wrote and reads: only the LDS counter needs to drain
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
#pragma unroll
        for (int p = 0; p < MIS * 4; ++p) {
            const int row = p * 8 + (lane >> 3), unit = lane & 7;
            const u32x4 v = *reinterpret_cast<const u32x4 *>(tile + row * 64 + ((unit ^ (row & 7)) << 3));
            const int grow = m0 + row_first + row;
            if (grow < M)
                *reinterpret_cast<u32x4 *>(C + (size_t)grow * N + n0 + wn * 64 + unit * 8) = v;
        }
    }
    KILN_TL(5);
}

}  // namespace

#ifdef KILN_PREFILL_TIMELINE
extern "C" int kiln_w4a16_debug_timeline(long long *buf) {
    return (int)hipMemcpyToSymbol(HIP_SYMBOL(g_timeline), &buf, sizeof(buf));
}
#endif

size_t prefill_aext_bytes(int m, int k) { return (size_t)m * (k / kGroupK) * sizeof(u32x4); }

// Scratch of the projection.  For the small-M kernels (few_rows): up to 16 K slices of T in bf16.
// For the matrix-core kernel: T once and behind it the f32 tiles in which the slices meet (at most
// ceil(256 / row tiles) slices per row tile: fewer than 256 + 2 x row tiles tiles of 64 or 16 rows
// x 64 columns).
constexpr int kProjectMaxCounters = (int)(kWsCounterCapacity / sizeof(int));  // the counter region less its sticky word
constexpr int kProjectFoldCounters = 8192;  // folded into the product's launch: the product's counters first, then the projection's
// measured at 2048 rows: 16-row blocks 9.9 us against 13.1 for K = 2560, 23.5 against 20.2 for K = 9216
int lora_project_rows_per_block(int m, int k) { return m > 1024 && k > 4096 ? 64 : 16; }
int prefill_lora_max_slices(int) { return 16; }
size_t prefill_lora_t_bytes(int m, bool few_rows) {
    if (few_rows) return (size_t)prefill_lora_max_slices(m) * m * 64 * sizeof(uint16_t);
    size_t many = 0;
    for (int rb = 16; rb <= 64; rb *= 4) {  // either block height
        const size_t tiles = 256 + 2 * (size_t)((m + rb - 1) / rb);
        const size_t bytes = (size_t)m * 64 * sizeof(uint16_t) + tiles * rb * 64 * sizeof(float);
        if (bytes > many) many = bytes;
    }
    return many;
}

// Rows of the die grid (a power of two up to 8; the dies form rows x 8 / rows over row blocks x units): the one
// under which the busiest die has the least to do -- ceil(row blocks / rows) row blocks of ceil(units / columns)
// units each, a whole tile counting as `ks` slices -- and of equals the one with the most rows, so that a die
// keeps few row blocks of A in its L2.  Neither count need divide: the grid is padded with blocks that leave at once.
// (Until the row blocks could be padded it was the largest power of two that divides them, i.e. one row of
// eight columns for any odd count, which leaves dies idle wherever the units are fewer than eight or do not
// divide by eight: 1024 -> 1024 at 20000 rows, 313 row blocks of three whole column blocks and one more, ran
// 165 us on three dies and then one, against 58 us at 19968 rows.)
//
// 0: no grid -- whole tiles that are no more than the compute units, where every grid leaves a die more of them than it has
// units (13 row blocks x 18 column blocks: 36 on six dies of 32 units): they are dealt one after the other, the row blocks
// of a column block first, and every die gets the same number.  (A second round of a few blocks each, and no second set of
// wavefronts: 3584 -> 4608 at 777 rows 58 -> 42 us, 4096 -> 3584 at 1100 64 -> 43, 18944 -> 3584 at 1100 233 -> 163; 128-row
// blocks, 4096 -> 2560 at 3200 rows 93 -> 67, 9216 -> 2560 at 3200 201 -> 140.)
static int prefill_die_rows(int m_blocks, int units_full, int units_sliced, int ks, int cus) {
    int best = 1;
    long best_work = -1;
    for (int dr = 8; dr >= 1; dr >>= 1) {
        const int dc = 8 / dr, rows = (m_blocks + dr - 1) / dr;
        const long work = (long)rows * ((long)((units_full + dc - 1) / dc) * ks + (units_sliced + dc - 1) / dc);
        if (best_work < 0 || work < best_work) {
            best = dr;
            best_work = work;
        }
    }
    if (units_sliced == 0 || (units_full == 0 && ks == 1)) {
        const int dc = 8 / best, units = units_full + units_sliced;
        const long tiles = (long)m_blocks * units, on_a_die = (long)((m_blocks + best - 1) / best) * ((units + dc - 1) / dc);
        if (8 * on_a_die > cus && (tiles + 7) / 8 * 8 <= cus) return 0;
    }
    return best;
}
static int prefill_die_rows(int m_blocks, int n, const PrefillPlan &p, int cus) {
    return prefill_die_rows(m_blocks, p.nb_full, (n / p.bn - p.nb_full) * p.ks, p.ks, cus);
}

// blocks launched: whole tiles, then (tile, K slice) units, each part padded to the die grid
int prefill_grid(int m, int n, const PrefillPlan &p, int cus) {
    const int m_blocks = (m + p.bm - 1) / p.bm;
    const int dr = prefill_die_rows(m_blocks, n, p, cus);
    if (dr == 0) return (m_blocks * (n / p.bn) + 7) / 8 * 8;
    const int dc = 8 / dr, rows = (m_blocks + dr - 1) / dr;
    const int units_full = p.nb_full, units_sliced = (n / p.bn - p.nb_full) * p.ks;
    return 8 * rows * ((units_full + dc - 1) / dc) + 8 * rows * ((units_sliced + dc - 1) / dc);
}

// Whole-tile part and K slices for a block shape.  Whole rounds of tiles (one tile per
// compute unit and round) run unsliced.  What is left -- everything, for a small problem --
// is cut into as many K slices as still leave one block per compute unit and three groups
// per slice, so the last round is as full as the others instead of leaving most of the chip
// idle.
static PrefillPlan plan_for_shape(int m, int n, int k, int cus, int bn, int bm, int sliced_units = 0) {
    if (sliced_units <= 0) sliced_units = cus;  // (tile, K slice) units the sliced round may have
    PrefillPlan p;
    p.bn = bn;
    p.bm = bm;
    const int G = k / kGroupK, m_blocks = (m + bm - 1) / bm;
    const int n_blocks = n / bn, tiles = m_blocks * n_blocks;
    const int rounds = tiles / cus;
    p.nb_full = (rounds * cus) / m_blocks;  // whole column blocks that fit the whole rounds
    if (p.nb_full > n_blocks) p.nb_full = n_blocks;
    // ... on every die: the dies deal the tiles as a grid (prefill_die_rows), and a die whose rectangle holds more
    // whole tiles than its share of the rounds runs a round of its own behind them (4096 -> 4096 at 1100 rows: 18
    // row blocks x 14 column blocks are 252 tiles, but 36 on each of six dies of 32 units -- 80 us, against 62 us at
    // 1217 rows, whose 20 x 12 are 30 per die)
    for (;; --p.nb_full) {
        const int rest = n_blocks - p.nb_full;
        p.ks = 1;
        for (int ks = 2; ks <= 8 && G / ks >= 3; ++ks) {
            const int gsb = (G + ks - 1) / ks;
            if ((ks - 1) * gsb >= G) continue;  // would leave an empty slice
            const int dr = prefill_die_rows(m_blocks, p.nb_full, rest * ks, ks, 0), dc = 8 / dr;
            if (8 * ((m_blocks + dr - 1) / dr) * ((rest * ks + dc - 1) / dc) <= sliced_units) p.ks = ks;
        }
        if (p.nb_full == 0 || p.nb_full == n_blocks) break;
        const int dr = prefill_die_rows(m_blocks, p.nb_full, rest * p.ks, p.ks, 0), dc = 8 / dr;
        if (((m_blocks + dr - 1) / dr) * ((p.nb_full + dc - 1) / dc) <= rounds * (cus / 8)) break;
    }
    return p;
}

// Relative cost of a plan in units of one 128-column block's group: whole rounds, then the
// sliced round, then the exchange of its partial tiles (wider blocks take about 1.3 times as
// long per group and exchange twice the data).
// A 128-row block takes 1.5 times as long per group as a 64-row one, exchanges at four times the price per
// slice, and its launch carries 6 units more (the row sums from a launch in front, a longer prologue and
// store): fitted to 98 cases -- 14 shapes at 400 ... 4096 rows, each with 64- and 128-row blocks forced --
// and to 72 more -- 12 shapes of other models at 129 ... 512 rows, the three block shapes forced -- on which
// the cheaper plan by this cost was the faster one or within 0.8 % (the former) and 0.6 % (the latter) of it
// on average, 18 % and 5 % at worst.  That was before the main loop was ordered by hand; on the kernel as it is, 88
// cases -- eight shapes at 200 ... 2048 rows, both heights forced -- are 2.4 % off on average and 32 % at worst
// (4096 -> 12288 at 420 rows: 62 us in 128-row blocks and two slices, 47 in 64-row ones).  With two sets of wavefronts to
// lone blocks and the rules behind the choice (plan_prefill), 233 cases -- 22 shapes at 192 ... 2048 rows, both heights in
// every number of slices -- are about 1 % off on average, 23 % at worst (6144 -> 6144 at 1300 rows, 64-row blocks in whole
// rounds and a rest: 124 us, whole 101).
static float plan_cost(int m, int n, int k, int cus, const PrefillPlan &p) {
    const int G = k / kGroupK, m_blocks = (m + p.bm - 1) / p.bm, n_blocks = n / p.bn;
    const float rows = p.bm == 128 ? 1.5f : 1.0f;
    const float per_group = (p.bn == 256 ? 1.3f : 1.0f) * rows;
    const float per_slice = (p.bm == 128 ? 2.0f : 0.5f) * rows;
    float cost = (float)((m_blocks * n_blocks) / cus) * G * per_group + (p.bm == 128 ? 6.f : 0.f);
    if (n_blocks > p.nb_full) {
        cost += (float)((G + p.ks - 1) / p.ks) * per_group;
        if (p.ks > 1) cost += per_slice * p.ks;
        // 128-row blocks sit two to a unit: behind whole rounds, the blocks of a K-sliced rest run beside the last round's
        // and hold it up by their own length, in proportion to how many of them there are (gate+up at 640
        // rows, 255 whole tiles and 105 in two slices of ten groups: 87.5 us, 73 with every tile whole or in
        // 64-row blocks; at 512 rows, 32 tiles in five slices of four groups: nothing)
        // (0.75 of that, and nothing for a rest of whole tiles, which is a round like the others: fitted with the rest)
        if (p.bm == 128 && p.nb_full > 0 && p.ks > 1)
            cost += 0.75f * (float)((n_blocks - p.nb_full) * m_blocks * p.ks) / cus * ((G + p.ks - 1) / p.ks) * per_group;
    }
    return cost;
}

// Block shape for a problem.  64-row blocks (four wavefronts side by side, three blocks per compute
// unit) for small problems, which are bound by latency and by how evenly the tiles cover the chip,
// not by the matrix cores (rows past M are computed and dropped); 128 x 256 blocks (four wavefronts
// side by side, each 128 x 64) where the chip is saturated: the best measured rate, because every
// wavefront's weights are its own and A is shared by all four.  Which of the two, and which width
// of the 64-row block: the lower modelled cost (plan_cost); up to 128 rows always 64 (until the 129...512-row
// sweep it was 384, and 128 x 256 blocks in K slices were missed where they lead by 15...25 %: 18944 -> 3584 at
// 321 rows 81.5 us against 107, 28672 -> 8192 at 256 rows 150 against 173, 6144 -> 6144 at 321 rows 51 against 68).  (A fixed
// switch at 768 rows was 5 % slower on average over the same 98 cases and 69 % at worst: narrow
// outputs want 64 rows at any row count, large products 128 rows from 400 on.)
// The 256-row shapes stay available through the overrides.
PrefillPlan plan_prefill(int m, int n, int k, int cus, int force_bn, int force_bm) {
    // 128-row tiles for 50...100 % of the compute units: two such blocks fit a unit, and with every tile cut
    // into as many K slices as fill those slots the chip is busier than with 64-row blocks, provided a slice
    // stays long (measured on N = 2560: K = 9216 at M = 2048 / 2560 / 3072, three or two slices of 24 or 36
    // groups, 121 / 148 / 162 us against 124 / 159 / 168; K = 4096 at M = 3072 in two slices of 16 groups
    // 90 against 84)
    int sliced_units = 0;
    {
        const int tiles = ((m + 127) / 128) * (n / 256);
        if (2 * tiles >= cus && tiles < cus) {
            const int ks = 2 * cus / tiles;
            // (shorter slices where the tiles leave a quarter of the units idle or more: 160 tiles of 8192 -> 10240 at
            // 448...512 rows in three slices of 21 / 22 groups 103.5 us against 119 in two and 114...125 in 64-row
            // blocks; 128 tiles of 8192 -> 8192, 14336 -> 8192, 28672 -> 8192 in four slices 3...8 % ahead of two)
            const int min_groups = 4 * tiles <= 3 * cus ? 16 : 24;
            if (ks >= 2 && k / kGroupK / ks >= min_groups) sliced_units = 2 * cus;
        }
    }
    if (force_bm == 64 || force_bm == 128 || force_bm == 256) {
        const int bm = force_bm;
        if (force_bn == 128 || force_bn == 256) return plan_for_shape(m, n, k, cus, force_bn, bm);
        const PrefillPlan wide = plan_for_shape(m, n, k, cus, 256, bm, bm == 128 ? sliced_units : 0);
        if (bm == 128) return wide;
        const PrefillPlan narrow = plan_for_shape(m, n, k, cus, 128, bm);
        if (bm == 64) return plan_cost(m, n, k, cus, narrow) <= plan_cost(m, n, k, cus, wide) ? narrow : wide;
        // 256-row blocks: narrow unless its tiles neither fill a round nor can be sliced
        if (narrow.nb_full == 0 && narrow.ks == 1 && wide.nb_full == 0 && wide.ks >= 2) return wide;
        return narrow;
    }
    // 64-row blocks of either width, and from 385 rows on 128 x 256 blocks: whichever the cost model prices lower
    PrefillPlan best = plan_for_shape(m, n, k, cus, force_bn == 128 ? 128 : 256, 64);
    if (force_bn != 128 && force_bn != 256) {
        const PrefillPlan narrow = plan_for_shape(m, n, k, cus, 128, 64);
        // (not as whole rounds plus a rest in five slices or more: 4096 -> 12288 at 129...192 rows ran 70.7 us as
        // 85 whole column blocks and 11 in seven slices against 47.4 as 64 x 256 blocks, 6144 -> 6144 at 321 rows
        // 103 against 68.5)
        const bool rest_in_many_slices = narrow.nb_full > 0 && narrow.ks >= 5;
        // Two wavefronts a block: for outputs too narrow to give the wider block enough tiles (2560 -> 1024 at
        // 400...4096 rows 17...36 us against 27...43).  On wider outputs the model's 1.0 : 1.3 a group does not hold
        // where a compute unit gets one such block (3584 -> 4608 at 448 rows, 252 tiles: 65 us, 38...44 in the other
        // shapes), and over 170 forced cases it never led by more than 3 % there.
        const bool narrow_output = n <= 2048;
        if (narrow_output && !rest_in_many_slices && plan_cost(m, n, k, cus, narrow) <= plan_cost(m, n, k, cus, best))
            best = narrow;
    }
    if (m > 128 && force_bn != 128) {
        const PrefillPlan tall = plan_for_shape(m, n, k, cus, 256, 128, sliced_units);
        if (plan_cost(m, n, k, cus, tall) < plan_cost(m, n, k, cus, best)) best = tall;
    }
    // 128-row tiles that would be cut in two slices, which sit two to a unit: whole where a unit's two sets of wavefronts can
    // share them, which needs no exchange (us, two slices -> whole: 4096 -> 4096 at 1300 / 1536 rows 61 -> 54 / 62 -> 55,
    // 9216 -> 2560 at 2300 / 2560 / 3072 rows 119 -> 113 / 124 -> 117 / 141 -> 137, 8192 -> 8192 at 768 rows 108 -> 101, 13824 -> 5120 at 1280
    // rows 177 -> 168; 14 shapes and row counts, the least 1 %, 18944 -> 3584 at 2048 rows).  Tiles for fewer than two thirds
    // of the units stay in three slices: 160 tiles of 8192 -> 8192 at 640 rows 88 in three, 97 whole, of 14336 -> 4096 at
    // 1280 rows 143 against 161.
    if (best.bm == 128 && best.bn == 256 && best.nb_full == 0 && best.ks == 2) {
        PrefillPlan whole = best;
        whole.nb_full = n / 256;
        whole.ks = 1;
        if (3 * ((m + 127) / 128) * (n / 256) >= 2 * cus && prefill_halves_k(m, n, k, whole, cus)) return whole;
    }
    // Three slices or more of 128-row tiles, of at most 16 groups, beyond 512 rows: as many of 64-row tiles, two blocks to a
    // unit, where these sum their rows themselves.  The taller blocks' short main loop waits for the blocks that form the row
    // sums, one per 16 rows (us, 128 -> 64 rows: 4096 -> 2560 at 777 / 900 / 1000 rows 35.1 -> 32.2 / 35.5 -> 32.8 / 36.1 -> 34.4,
    // 4096 -> 4096 at 640 36.5 -> 33.2, 3072 -> 2560 at 777 30.8 -> 26.9, 6144 -> 2560 at 1000 46.5 -> 44.8, the least; 51
    // shapes and row counts, 4 to 13 %.  At 450 and 512 rows it is level to 9 %, 5120 -> 4608 2 % behind; in longer shares
    // level, 9216 -> 2560 at 900).
    if (best.bm == 128 && best.bn == 256 && best.nb_full == 0 && best.ks >= 3 && m > 512 &&
        (k / kGroupK + best.ks - 1) / best.ks <= 16 && !prefill_halves_k(m, n, k, best, cus)) {
        PrefillPlan low = best;
        low.bm = 64;
        const int grid = prefill_grid(m, n, low, cus);
        if (grid > cus && grid <= 2 * cus && prefill_rowsum_producers(m, n, k, low, cus) == -2) return low;
    }
    return best;
}
size_t prefill_partial_bytes(int m, int n, const PrefillPlan &p) {
    if (p.ks <= 1) return 0;
    return (size_t)((m + p.bm - 1) / p.bm) * p.bm * (size_t)(n - p.nb_full * p.bn) * p.ks * sizeof(float);
}

namespace {

// Bytes of LDS for the in-kernel row sums of a 64-row block covering `groups` groups of K.
constexpr int kMaxRowSumBytes = 24 * 1024;
static int row_sum_bytes(int groups) { return groups * 64 * (int)sizeof(float); }


template <int NWN, int WM, int MI, bool SWIGLU, bool RS, bool FOLD = false, bool INC = false, int WK = 1>
hipError_t launch_shape_as(const PrefillArgs &a, int grid, int m_blocks, int RP, int KS, int GSb, int max_groups,
                           hipStream_t stream, const PrefillFold &pf = PrefillFold{}) {
    constexpr int BM = WM * MI * 32, NW = WM * NWN;
    // the A rings, behind them the groups' c or the extension's scales
    constexpr int kRing = WK * (kAStages * BM * 64 + (INC ? 2 * NW * 256 : RS ? 0 : kAStages * NW * 512)) + (WK == 2 && FOLD ? 1024 : 0);
    // the store's per-wavefront transposes, or twice that where the halves of K meet (reuses the rings)
    constexpr int kStore = NW * MI * 32 * 64 * 2 * WK;
    // RS: the row sums sit behind the ring and are dead by the time the store reuses the space
    constexpr int kLdsMax = RS ? (kRing + kMaxRowSumBytes + 256 > kStore ? kRing + kMaxRowSumBytes + 256 : kStore)
                               : (kRing > kStore ? kRing : kStore);
    int lds_bytes = kRing > kStore ? kRing : kStore;
    const int sums = row_sum_bytes((max_groups + WK - 1) / WK * WK);  // (each half of K: its own groups')
    if (RS && kRing + sums > lds_bytes) lds_bytes = kRing + sums;
    // The 256 x 128 block fits twice on a compute unit.  A grid of at most one block per unit
    // asks for more LDS than two blocks could share, so the dispatcher cannot stack two blocks
    // on one unit while others idle.
    constexpr int kLdsSolo0 = (WM == 2 && NWN == 2) ? 96 * 1024 : kLdsMax;
    constexpr int kProjectLds = WK == 2 ? stream_lds_bytes(32, RS ? 0 : kStreamMaxSums) : kProjectLdsBytes16;
    constexpr int kLdsSolo = FOLD && kLdsSolo0 < kProjectLds ? kProjectLds : kLdsSolo0;
    const hipError_t attr = allow_dynamic_lds<&w4a16_prefill_kernel<NWN, WM, MI, SWIGLU, RS, FOLD, INC, WK>>(kLdsSolo);
    if (attr != hipSuccess) return attr;
    if (WM == 2 && NWN == 2 && grid <= a.cus) lds_bytes = kLdsSolo;
    // the projection's blocks stage more
    const int project_lds = WK == 1 ? kProjectLdsBytes16
                            : pf.a_cat ? stream_lds_bytes(RP, RS ? 0 : pf.steps_per_slice / 4) : 0;
    if (FOLD && lds_bytes < project_lds) lds_bytes = project_lds;
    w4a16_prefill_kernel<NWN, WM, MI, SWIGLU, RS, FOLD, INC, WK><<<grid + (FOLD ? pf.producers : 0), 64 * NW * WK, lds_bytes, stream>>>(
        (const uint16_t *)a.A, (const u32x4 *)a.B, (const uint16_t *)a.S, (uint16_t *)a.C, (const u32x4 *)a.aext,
        a.M, a.N, a.K, a.Gs, m_blocks, (const uint16_t *)a.lora_t, (const uint16_t *)a.lora_b, a.r_total, RP,
        a.nb_full, KS, GSb, a.partial, a.counters,
        prefill_die_rows(m_blocks, a.nb_full, (a.N / (NWN * 64) - a.nb_full) * KS, KS, a.cus), (u32x4 *)a.next_aext, a.next_plain, pf);
    return hipGetLastError();
}

template <int NWN, int WM, int MI, int WK = 1>
hipError_t launch_shape(const PrefillArgs &a, int grid, int m_blocks, int RP, int KS, int GSb, int max_groups,
                        bool rs, hipStream_t stream) {
    if constexpr (MI == 2) {
        if (rs)
            return a.swiglu ? launch_shape_as<NWN, WM, MI, true, true, false, false, WK>(a, grid, m_blocks, RP, KS, GSb, max_groups, stream)
                            : launch_shape_as<NWN, WM, MI, false, true, false, false, WK>(a, grid, m_blocks, RP, KS, GSb, max_groups, stream);
    }
    return a.swiglu ? launch_shape_as<NWN, WM, MI, true, false, false, false, WK>(a, grid, m_blocks, RP, KS, GSb, max_groups, stream)
                    : launch_shape_as<NWN, WM, MI, false, false, false, false, WK>(a, grid, m_blocks, RP, KS, GSb, max_groups, stream);
}

// A launch whose first blocks write what the others need (PrefillFold): blocks of 256 columns.
template <int MI, int WK>
hipError_t launch_fold(const PrefillArgs &a, int grid, int m_blocks, int RP, int KS, int GSb, int max_groups, bool rs,
                       const PrefillFold &pf, hipStream_t stream) {
    if constexpr (MI == 2) {
        if (rs)
            return a.swiglu ? launch_shape_as<4, 1, MI, true, true, true, false, WK>(a, grid, m_blocks, RP, KS, GSb, max_groups, stream, pf)
                            : launch_shape_as<4, 1, MI, false, true, true, false, WK>(a, grid, m_blocks, RP, KS, GSb, max_groups, stream, pf);
    }
    return a.swiglu ? launch_shape_as<4, 1, MI, true, false, true, false, WK>(a, grid, m_blocks, RP, KS, GSb, max_groups, stream, pf)
                    : launch_shape_as<4, 1, MI, false, false, true, false, WK>(a, grid, m_blocks, RP, KS, GSb, max_groups, stream, pf);
}

// A launch that adds the row sums at the groups' changes (INC): blocks of 128 rows and 256 columns.
template <bool FOLD, int WK>
hipError_t launch_sums_in_loop(const PrefillArgs &a, int grid, int m_blocks, int RP, int KS, int GSb, int max_groups,
                               const PrefillFold &pf, hipStream_t stream) {
    return a.swiglu ? launch_shape_as<4, 1, 4, true, false, FOLD, true, WK>(a, grid, m_blocks, RP, KS, GSb, max_groups, stream, pf)
                    : launch_shape_as<4, 1, 4, false, false, FOLD, true, WK>(a, grid, m_blocks, RP, KS, GSb, max_groups, stream, pf);
}

}  // namespace

// K slices of the projection for few rows (the small-M kernels multiply T): up to 16, each staging
// two pieces; the consumer runs over them as if they were further rank columns, which costs it
// less than a meeting of the blocks would cost here.
int lora_project_slices(int m, int k) {
    const int pieces = (k + kProjectPieceK - 1) / kProjectPieceK;
    int kz = (pieces + 1) / 2;
    if (kz > prefill_lora_max_slices(m)) kz = prefill_lora_max_slices(m);
    return kz < 1 ? 1 : kz;
}

// Many rows, `rb` a block: row tiles, K slices (as many as keep about 256 blocks busy, at most `most`) and steps of
// 32 values per slice (whole groups).
struct ProjectSlicing {
    int row_tiles, kz, per_slice;
};
static ProjectSlicing project_slicing(int m, int k, int rb, bool have_counters, int most) {
    const int steps = k / 32, row_tiles = (m + rb - 1) / rb;
    const int pieces = (k + kProjectPieceK - 1) / kProjectPieceK;
    int kz = (256 + row_tiles - 1) / row_tiles;
    const int zmax = rb == 16 ? 16 : 8;  // what the kernel's meeting reads in one go
    if (kz > zmax) kz = zmax;
    if (kz > pieces) kz = pieces;
    if (row_tiles > kProjectMaxCounters || !have_counters) kz = 1;
    if (kz > most) kz = most;
    const int per_slice = ((steps + kz - 1) / kz + 3) / 4 * 4;
    return {row_tiles, (steps + per_slice - 1) / per_slice, per_slice};
}

// `kz`, `per_slice` (many rows): the K slices of a projection that could run inside the product's launch, whose sums it
// then adds in the same order; 0: as many as suit a launch of its own.
static hipError_t project_in_front(const PrefillArgs &a, bool few_rows, hipStream_t stream, int *slices, bool with_row_sums,
                                   bool plain_sums, int kz, int per_slice) {
    if (a.r_total < 1 || a.r_total > kProjectMaxRank || a.n_adapters < 1 || a.n_adapters > 8 || !a.lora_a ||
        !a.lora_t || !a.ranks || !a.scales || a.M < 1 || a.K < kGroupK)
        return hipErrorInvalidValue;
    const int RP = (a.r_total + 15) / 16 * 16;
    LoraScales ls;
    ls.count = a.n_adapters;
    int end = 0;
    for (int i = 0; i < 8; ++i) {
        if (i < a.n_adapters) end += a.ranks[i];
        ls.ends[i] = end;
        ls.scales[i] = i < a.n_adapters ? a.scales[i] : 0.f;
    }
    *slices = 1;
    const int steps = a.K / 32;
    u32x4 *aext = with_row_sums && !few_rows ? (u32x4 *)a.aext : nullptr;
    if (with_row_sums && !aext) return hipErrorInvalidValue;
    if (!few_rows) {
        // many rows: T whole.  K slices that meet in f32 behind T, as many as keep about 256 blocks busy.
        const int rb = lora_project_rows_per_block(a.M, a.K);
        const ProjectSlicing own = project_slicing(a.M, a.K, rb, a.counters != nullptr, INT_MAX);
        const int row_tiles = own.row_tiles;
        if (kz == 0 || row_tiles > kProjectMaxCounters || !a.counters) {
            kz = own.kz;
            per_slice = own.per_slice;
        }
        float *partial = reinterpret_cast<float *>(reinterpret_cast<char *>(a.lora_t) + (size_t)a.M * 64 * sizeof(uint16_t));
        const int lds_bytes = (rb + kProjectMaxRank) * kProjectRowBytes + kProjectMaxRank * (int)sizeof(float);
        const auto kernel = rb == 16 ? (plain_sums ? &w4a16_lora_project_kernel<16, true> : &w4a16_lora_project_kernel<16, false>)
                                     : (plain_sums ? &w4a16_lora_project_kernel<64, true> : &w4a16_lora_project_kernel<64, false>);
        if (rb == 64) {
            const hipError_t attr = plain_sums ? allow_dynamic_lds<&w4a16_lora_project_kernel<64, true>>(lds_bytes)
                                               : allow_dynamic_lds<&w4a16_lora_project_kernel<64, false>>(lds_bytes);
            if (attr != hipSuccess) return attr;
        }
        kernel<<<dim3(row_tiles, kz), 256, lds_bytes, stream>>>(
            (const uint16_t *)a.A, (const uint16_t *)a.lora_a, (uint16_t *)a.lora_t, a.M, a.K, a.r_total, RP, per_slice, ls, partial,
            a.counters, aext);
        return hipGetLastError();
    }
    kz = lora_project_slices(a.M, a.K);
    per_slice = ((steps + kz - 1) / kz + 3) / 4 * 4;  // whole 128-value groups
    kz = (steps + per_slice - 1) / per_slice;
    *slices = kz;
    const int lds_bytes = (16 + kProjectMaxRank) * kProjectRowBytes + kProjectMaxRank * (int)sizeof(float);
    w4a16_lora_project_kernel<16, false><<<dim3((a.M + 15) / 16, kz), 256, lds_bytes, stream>>>(
        (const uint16_t *)a.A, (const uint16_t *)a.lora_a, (uint16_t *)a.lora_t, a.M, a.K, a.r_total, RP, per_slice, ls,
        nullptr, nullptr, nullptr);
    return hipGetLastError();
}

hipError_t launch_lora_project(const PrefillArgs &a, bool few_rows, hipStream_t stream, int *slices, bool with_row_sums,
                               bool plain_sums) {
    return project_in_front(a, few_rows, stream, slices, with_row_sums, plain_sums, 0, 0);
}

// 64-row blocks form the row sums themselves when they fit next to the A ring and the launch is
// bound by latency rather than by work (measured: -2...-10 % up to about 28 GFLOP or on narrow
// outputs, +6...+8 % beyond, where the extra VALU and LDS work in the main loop costs more
// than the saved pre-pass launch)
static bool blocks_sum_their_rows(int M, int N, int K, const PrefillPlan &p) {
    const int G = K / kGroupK, ks = p.ks < 1 ? 1 : p.ks;
    // most groups of K any one block covers: all of them for a whole tile
    const int max_groups = p.nb_full > 0 ? G : (G + ks - 1) / ks;
    const double flops = 2.0 * M * (double)N * K;
    return p.bm == 64 && row_sum_bytes(max_groups) <= kMaxRowSumBytes && (flops <= 28e9 || N <= 4096);
}

// Row-sum producers a launch should have: one per 64 rows, in eights.
static int rowsum_producers_wanted(int M) { return ((M + 63) / 64 + 7) / 8 * 8; }

// Blocks whose wavefronts share K (the kernel's WK): where the plan gives a compute unit one block at most, of enough groups
// that half of them pay for the halves' meeting.  The row sums: from the blocks, from the units without a block where they
// can be done in time, else, for whole tiles, from a launch in front, which 128-row blocks then add at the changes of group.
// By the plan alone, with adapters or without, and alike for both block widths (counted in blocks of 256 columns), so that calls
// which must agree in every bit add in one order.  (Plain calls, 70 shapes of 200 ... 1300 rows, 1024 ... 9216 wide: 1.11 times
// as fast on average, those that take it 1 % slower at worst.  Calls with adapters, whose projection runs beside the blocks or
// in front, project_place: 1.06 times as fast on average, 0.86 at worst, 5 of 70 below 0.97.  Where it is not taken: shorter
// shares are level or slower, 11 groups in 128-row blocks, 4096 -> 2560 at 777 rows in three slices, 33.7 us either way; 64-row
// blocks on every unit, 2816 -> 1024 at 2000 rows, 256 blocks of 11 groups, and 2048 -> 2048 at 900, 2 to 7 % slower: the units'
// store and start then have nothing left to hide behind.  128-row blocks of fewer than 24 groups gain 3.5 % plain and lost 5 to
// 11 % with adapters, 2560 -> 8192 at 777 rows 44 -> 50 us.  With the sums from a launch in front, tiles for nine tenths of the
// units or all: 4096 -> 4096 at 1900 / 2048 rows 74 -> 67 us, 4096 -> 2560 at 3072 82 -> 75, 8192 -> 8192 at 1024 133 -> 123,
// 14336 -> 4096 at 2048 228 -> 213, 28672 -> 8192 at 1000 470 -> 415, 3072 -> 8192 at 1000 54.3 -> 53.0, the least.  Launches of
// several rounds are slower so: 2560 -> 18432 at 777 / 4096 rows 72 -> 80 / 307 -> 343, one block of eight wavefronts a unit in place
// of two of four.)
bool prefill_halves_k(int M, int N, int K, const PrefillPlan &p, int cus) {
    if ((p.bm != 64 && p.bm != 128) || p.nb_full < 0 || p.nb_full > N / p.bn) return false;
    const int G = K / kGroupK, ks = p.ks < 1 || p.nb_full == N / p.bn ? 1 : p.ks;  // (of whole tiles alone: nothing is sliced)
    PrefillPlan wide = p;
    wide.bn = 256;
    wide.nb_full = p.nb_full * p.bn / 256;
    const int grid = prefill_grid(M, N, wide, cus), row_tiles = (M + 15) / 16;
    if (grid > cus || (G + ks - 1) / ks < (p.bm == 128 ? 24 : grid <= cus - 8 ? 6 : 16)) return false;
    if (blocks_sum_their_rows(M, N, K, p)) return true;
    // the producers' share must be done before a block's main loop is: 0.7 ns a row tile and value of K against
    // 1.4 us a group
    const int producers = (cus - grid) / 8 * 8;
    if (row_tiles > kPrefillFoldMaxTiles || producers < rowsum_producers_wanted(M)) return ks == 1;  // (from a launch in front)
    return (row_tiles + producers - 1) / producers * ks <= 11;
}

// Without adapters a few of the product's own first blocks form the row sums (rowsum_producer_block)
// where the launch is a single round of blocks that leaves block slots free: producers in those
// slots cost the product nothing and save the launch in front (down projection at 2048 rows
// 116 -> 112 us, 2560 -> 8192 at 777 rows 61 -> 59.5).  They must be done before the first block's main
// loop is: at least one per 64 rows (its piece of A then streams in about half that time, whatever
// K), as many as there are free slots up to one per 16-row tile.  In a launch of several rounds the
// producers' slots are taken from the product: measured 2 to 5 us slower than the launch in front
// (gate+up at 2048 and 4096 rows), so those keep it.  0: from the launch in front; -2: the blocks sum
// their rows themselves.
int prefill_rowsum_producers(int M, int N, int K, const PrefillPlan &p, int cus) {
    if (blocks_sum_their_rows(M, N, K, p)) return -2;
    if (p.bn != 256 || (p.bm != 64 && p.bm != 128) ||
        (M + 15) / 16 > kPrefillFoldMaxTiles || p.nb_full < 0 || p.nb_full > N / p.bn)
        return 0;
    const int grid = prefill_grid(M, N, p, cus), slots = cus * (prefill_halves_k(M, N, K, p, cus) ? 1 : p.bm == 128 ? 2 : 3);
    const int want = rowsum_producers_wanted(M), tiles8 = ((M + 15) / 16 + 7) / 8 * 8;
    const int free_slots = (slots - grid) / 8 * 8;
    if (free_slots < want) return 0;
    const int producers = free_slots < tiles8 ? free_slots : tiles8;
    return producers < 128 ? producers : 128;
}

// Where the row sums are added at the groups' changes (INC): 128-row blocks whose row sums prefill_rowsum_producers()
// leaves to a launch in front, with adapters and without.  By the shape alone, since the two routes of a shape's row
// sums must agree in every bit, and a call with adapters of zeros must equal the plain call.  Calls with overrides follow the
// automatic plan of their shape, also where they name blocks of 128 columns: the widths agree in every bit, and an override
// that changes nothing gives the automatic call's bits.  64-row blocks keep the extension contraction.
// (2560 -> 2 x 9216 -> 2560 at 8192 rows 933 -> 912 us, at 2048 rows 269 -> 260, error beyond the bf16 rounding 2.1e-4 -> 0.9e-4
// of the result's norm, 1.1e-3 -> 2.2e-4 where the activations have a mean of half their deviation: the surplus leaves group by
// group instead of piling up in the accumulators.  With two adapters, the projection inside the launch and the sums from the
// pre-pass kernel: 2560 -> 18432 at 1024 / 2048 / 4096 / 8192 rows 97.7 -> 98.3, 173.8 -> 172.8, 334 -> 327, 661 -> 650 us, error
// 1.6e-4 -> 0.7e-4; both from a launch in front: 101.6 at 1024 rows, 174.5 at 2048 where inside took 170.4.  Where the
// projection takes 64 rows a block, or finds no slots, it is in front and writes the sums: 9216 -> 2560 at 4096 rows 207 -> 200.)
bool prefill_adds_sums_in_loop(int M, int N, int K, const PrefillPlan &p, int cus) {
    return p.bn == 256 && p.bm == 128 && prefill_rowsum_producers(M, N, K, p, cus) == 0;
}
bool prefill_forms_next_sums(const PrefillPlan &p) { return p.bn == 256 && (p.bm == 64 || p.bm == 128); }
bool prefill_reads_row_sums(int M, int N, int K, const PrefillPlan &p) { return !blocks_sum_their_rows(M, N, K, p); }

// Where the projection of a call with adapters runs: in so many blocks in front of the product's in its launch, or (0) in a
// launch in front.
//
// A product that fits the chip's block slots in one go must still fit them with the projection's blocks
// in front: the blocks that find no slot start when the producers leave, on whichever units the
// dispatcher picks, and two of them on one unit beside idle units take 1.6 times as long as one (4096 ->
// 4096 at 1700 rows, 224 blocks of 128 x 256 and 328 producers for 512 slots: 121 us against 86 at 1600
// rows, 300 + 208 blocks; 97 with the projection in front).  So the projection is cut into fewer K slices
// there -- its blocks stay far shorter than the product's -- and runs in front if its row tiles alone do
// not fit.  Launches of several rounds keep all slices (gate+up at 2048 rows 189 us inside, 194 in front), and
// so do 64-row blocks, three to a unit, which were never seen to suffer (gate+up at 512 rows, 768 blocks and
// 256 producers for 768 slots: 62 us inside, 68 in front).
//
// Blocks whose wavefronts share K have a unit each, and the projection the units that are left (lora_project_stream), several
// shares one after the other where these are few.  In front where it would not be done in time: 0.4 us a group of K (0.8 with
// row sums) and 1.6 us a share against 1 us (128 rows: 1.2) a group of the product and 5 us around them.  Both places timed for
// 300 shapes and ranks of 180 ... 2048 rows: inside is 1.22 times as fast on average (2048 -> 6656 at 422 rows 29.9 -> 24.0 us), in
// front up to 1.8 times where a share is long (9216 -> 1280 at 1446 rows, two shares of 72 groups a block, 102 us inside, 66 in
// front); the rule is 0.04 % off the better of the two on average.  (us with one set of wavefronts in brackets: 1920 -> 3840
// at 648 rows 23.6 (26.8), 2944 -> 6400 at 291 29.5 (36.7), 7808 -> 2560 at 761 46.8 (55.3).  What stays in front, product
// launches of two or three K slices that leave 16 units or none, costs 6 us: 2048 -> 1280 at 1296 rows 27.5 (23.6).  Blocks of the
// projection placed where a die has most units left, instead of alike on all dies: 5 us slower.)
struct ProjectPlace {
    ProjectSlicing ps;
    int producers;
};
static ProjectPlace project_place(int M, int N, int K, const PrefillPlan &p, int cus, bool inc, bool have_counters) {
    const bool halves = prefill_halves_k(M, N, K, p, cus);
    const int rb = halves ? kFoldProjectRows<2> : lora_project_rows_per_block(M, K), G = K / kGroupK;
    ProjectPlace place{project_slicing(M, K, rb, have_counters, INT_MAX), 0};
    ProjectSlicing &ps = place.ps;
    if (p.bn != 256 || (p.bm != 64 && p.bm != 128) || (!halves && rb != 16) || (halves && inc)) return place;
    int producers = (ps.row_tiles * ps.kz + 7) / 8 * 8;
    if (halves || p.bm == 128) {
        const int slots = halves ? cus : cus * 2, product = prefill_grid(M, N, p, cus), left = (slots - product) / 8 * 8;
        if (product <= slots && producers > left) {
            if (left < (halves ? 1 : ps.row_tiles)) return place;
            ps = project_slicing(M, K, rb, have_counters, left >= ps.row_tiles ? left / ps.row_tiles : 1);
            producers = (ps.row_tiles * ps.kz + 7) / 8 * 8;
            if (producers > left) producers = left;
        }
    }
    if (halves) {
        const bool sums = prefill_reads_row_sums(M, N, K, p);
        const int share = ps.per_slice / (kGroupK / 32), turns = (ps.row_tiles * ps.kz + producers - 1) / producers;
        const int groups = p.nb_full > 0 || p.ks < 1 ? G : (G + p.ks - 1) / p.ks;
        const int needs = (sums ? 4 : 2) * share * turns + 8 * turns, has = (p.bm == 64 ? 5 : 6) * groups + 24;
        if ((sums && share > kStreamMaxSums) || needs > has) return place;
    }
    place.producers = producers;
    return place;
}
int prefill_projection_blocks(int M, int N, int K, const PrefillPlan &p, int cus) {
    return project_place(M, N, K, p, cus, prefill_adds_sums_in_loop(M, N, K, p, cus), true).producers;
}

hipError_t launch_prefill(const PrefillArgs &a, hipStream_t stream) {
    const int G = a.K / kGroupK;
    if (a.bm != 64 && a.bm != 128 && a.bm != 256) return hipErrorInvalidValue;
    const int KS_ = a.KS < 1 ? 1 : a.KS;
    PrefillPlan shape;
    shape.bn = a.bn;
    shape.bm = a.bm;
    shape.ks = KS_;
    shape.nb_full = a.nb_full;
    const int max_groups = a.nb_full > 0 ? G : (G + KS_ - 1) / KS_;
    const bool rs = blocks_sum_their_rows(a.M, a.N, a.K, shape);
    hipError_t err = hipSuccess;
    if (a.next_aext && !prefill_forms_next_sums(shape)) return hipErrorInvalidValue;
    const bool inc = a.sums_in_loop;
    if (inc && a.bm != 128) return hipErrorInvalidValue;
    const bool halves = prefill_halves_k(a.M, a.N, a.K, shape, a.cus);
    if (halves && !a.counters) return hipErrorInvalidValue;  // (the error word is at a fixed distance)
    const int inside = a.r_total == 0 && a.lora_words && !a.aext_ready && !inc ? prefill_rowsum_producers(a.M, a.N, a.K, shape, a.cus) : 0;
    const int sum_producers = inside > 0 ? inside : 0;
    int RP = 0;
    // The projection inside the product's launch (PrefillFold): four-wavefront blocks, 16-row tiles of T,
    // the extension operand from the projection (unless the blocks sum their rows themselves), and room
    // for its counters behind the product's.
    PrefillFold pf{};
    bool fold = false;
    if (a.r_total > 0) {
        RP = (a.r_total + 15) / 16 * 16;
        const ProjectPlace place = project_place(a.M, a.N, a.K, shape, a.cus, inc, a.counters != nullptr);
        const int row_tiles = (a.M + 15) / 16;
        const int sliced_tiles = (a.N / a.bn - a.nb_full) * ((a.M + a.bm - 1) / a.bm);
        fold = place.producers > 0 && a.lora_words && a.counters && row_tiles <= kPrefillFoldMaxTiles && row_tiles <= kProjectMaxCounters - kProjectFoldCounters &&
               sliced_tiles <= kProjectFoldCounters && a.n_adapters >= 1 && a.n_adapters <= 8 && a.lora_a && a.lora_t &&
               a.ranks && a.scales && a.r_total <= kProjectMaxRank;
        if (fold) {
            pf.a_cat = (const uint16_t *)a.lora_a;
            pf.t = (uint16_t *)a.lora_t;
            // blocks that sum their rows themselves need no operand, and with INC the sums have to be there
            // before a block begins
            pf.aext = rs || inc ? nullptr : (u32x4 *)a.aext;
            pf.partial = reinterpret_cast<float *>(reinterpret_cast<char *>(a.lora_t) + (size_t)a.M * 64 * sizeof(uint16_t));
            pf.counters = a.counters + kProjectFoldCounters;
            pf.words = a.lora_words;
            pf.row_tiles = row_tiles;
            pf.project_tiles = place.ps.row_tiles;
            pf.kz = place.ps.kz;
            pf.steps_per_slice = place.ps.per_slice;
            pf.producers = place.producers;
            pf.ls.count = a.n_adapters;
            int end = 0;
            for (int i = 0; i < 8; ++i) {
                if (i < a.n_adapters) end += a.ranks[i];
                pf.ls.ends[i] = end;
                pf.ls.scales[i] = i < a.n_adapters ? a.scales[i] : 0.f;
            }
        } else {
            int slices = 1;  // many rows: T is whole
            err = project_in_front(a, false, stream, &slices, !rs, inc, place.producers > 0 ? place.ps.kz : 0, place.ps.per_slice);
            if (err != hipSuccess) return err;
            if (slices != 1) return hipErrorInvalidValue;
        }
    }
    // with adapters the projection forms the row sums on its way over x, but for INC's where it runs inside the launch
    if (!rs && sum_producers == 0 && !a.aext_ready && (a.r_total == 0 || (inc && fold))) {
        const int items = a.M * G;
        (inc ? w4a16_prefill_rowsum_kernel<true> : w4a16_prefill_rowsum_kernel<false>)<<<(items + 15) / 16, 256, 0, stream>>>(
            (const uint16_t *)a.A, (u32x4 *)a.aext, a.M, a.K);
        err = hipGetLastError();
        if (err != hipSuccess) return err;
    }
    if (sum_producers > 0) {
        fold = true;
        pf.aext = (u32x4 *)a.aext;
        pf.words = a.lora_words;
        pf.row_tiles = (a.M + 15) / 16;
        pf.producers = sum_producers;
        pf.sum_tiles = (pf.row_tiles + sum_producers - 1) / sum_producers;
    }
    if (a.bn != 128 && a.bn != 256) return hipErrorInvalidValue;
    const int m_blocks = (a.M + a.bm - 1) / a.bm;
    const int KS = a.KS < 1 ? 1 : a.KS;
    const int GSb = (G + KS - 1) / KS;
    if (KS > 1 && (!a.partial || !a.counters || (KS - 1) * GSb >= G)) return hipErrorInvalidValue;
    if (a.nb_full < 0 || a.nb_full > a.N / a.bn) return hipErrorInvalidValue;
    const int grid = prefill_grid(a.M, a.N, shape, a.cus);
    if (fold) {
        pf.consumers = grid;
        if (inc)
            return launch_sums_in_loop<true, 1>(a, grid, m_blocks, RP, KS, GSb, max_groups, pf, stream);
        if (halves)
            return a.bm == 128 ? launch_fold<4, 2>(a, grid, m_blocks, RP, KS, GSb, max_groups, rs, pf, stream)
                               : launch_fold<2, 2>(a, grid, m_blocks, RP, KS, GSb, max_groups, rs, pf, stream);
        return a.bm == 128 ? launch_fold<4, 1>(a, grid, m_blocks, RP, KS, GSb, max_groups, rs, pf, stream)
                           : launch_fold<2, 1>(a, grid, m_blocks, RP, KS, GSb, max_groups, rs, pf, stream);
    }
    if (inc && a.bn == 128) {  // through overrides only, which the fused calls do not take
        if (a.swiglu) return hipErrorInvalidValue;
        return halves ? launch_shape_as<2, 1, 4, false, false, false, true, 2>(a, grid, m_blocks, RP, KS, GSb, max_groups, stream)
                      : launch_shape_as<2, 1, 4, false, false, false, true>(a, grid, m_blocks, RP, KS, GSb, max_groups, stream);
    }
    if (inc)
        return halves ? launch_sums_in_loop<false, 2>(a, grid, m_blocks, RP, KS, GSb, max_groups, pf, stream)
                      : launch_sums_in_loop<false, 1>(a, grid, m_blocks, RP, KS, GSb, max_groups, pf, stream);
    if (halves) {
        if (a.bm == 128)
            return a.bn == 256 ? launch_shape<4, 1, 4, 2>(a, grid, m_blocks, RP, KS, GSb, max_groups, rs, stream)
                               : launch_shape<2, 1, 4, 2>(a, grid, m_blocks, RP, KS, GSb, max_groups, rs, stream);
        return a.bn == 256 ? launch_shape<4, 1, 2, 2>(a, grid, m_blocks, RP, KS, GSb, max_groups, rs, stream)
                           : launch_shape<2, 1, 2, 2>(a, grid, m_blocks, RP, KS, GSb, max_groups, rs, stream);
    }
    if (a.bm == 256) {
        return a.bn == 256 ? launch_shape<4, 2, 4>(a, grid, m_blocks, RP, KS, GSb, max_groups, rs, stream)
                           : launch_shape<2, 2, 4>(a, grid, m_blocks, RP, KS, GSb, max_groups, rs, stream);
    } else if (a.bm == 128) {
        return a.bn == 256 ? launch_shape<4, 1, 4>(a, grid, m_blocks, RP, KS, GSb, max_groups, rs, stream)
                           : launch_shape<2, 1, 4>(a, grid, m_blocks, RP, KS, GSb, max_groups, rs, stream);
    }
    return a.bn == 256 ? launch_shape<4, 1, 2>(a, grid, m_blocks, RP, KS, GSb, max_groups, rs, stream)
                       : launch_shape<2, 1, 2>(a, grid, m_blocks, RP, KS, GSb, max_groups, rs, stream);
}

}  // namespace kiln
