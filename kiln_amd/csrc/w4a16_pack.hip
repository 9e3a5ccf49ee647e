// Quantise-and-pack on the device: bf16 weights [k, n] in device memory -> the tile layout of
// layout.h and its fp16 scales, without leaving the GPU.
//
// The arithmetic is the reference quantiser's (crates/kiln-marlin-gemm/src/lib.rs:393-427), as
// pack_host.cpp states it on the host, and the results are the same bits: per scale group and
// column s = f16(2 * max|w| / 15) (max == 0 -> 1.0), code = clamp(round(w / f32(s)) + 8, 0, 15) with
// ties away from zero and Rust's saturating float-to-int cast.  The reference has no device-side
// counterpart: marlin_proj.rs:86-181 downloads every weight, quantises on the host (17-58 s per
// model load for its 104 projections, ARCHITECTURE.md:570) and uploads the result.  Bound by memory
// traffic: 2 bytes read and half a byte written per weight.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kiln_w4a16.h"
#include "device_common.h"
#include "layout.h"

namespace kiln {
namespace {

// IEEE binary32 -> binary16, round to nearest even, in integer arithmetic (the host quantiser's
// f32_to_f16, half::f16::from_f32 at lib.rs:411): independent of the device's rounding and
// denormal modes.
__device__ uint16_t pack_f32_to_f16(float v) {
    const uint32_t x = __builtin_bit_cast(uint32_t, v);
    const uint16_t sign = (uint16_t)((x >> 16) & 0x8000u);
    const uint32_t ex = (x >> 23) & 0xFFu;
    uint32_t man = x & 0x7FFFFFu;
    if (ex == 0xFF) {
        if (!man) return sign | 0x7C00u;
        const uint16_t m = (uint16_t)(man >> 13);
        return sign | 0x7C00u | m | (m ? 0 : 0x0200u);
    }
    const int e = (int)ex - 112;
    if (e >= 31) return sign | 0x7C00u;
    if (e <= 0) {
        if (e < -10) return sign;
        man |= 0x800000u;
        const int shift = 14 - e;
        uint32_t h = man >> shift;
        const uint32_t rem = man & ((1u << shift) - 1u), half = 1u << (shift - 1);
        if (rem > half || (rem == half && (h & 1u))) ++h;
        return sign | (uint16_t)h;
    }
    uint32_t out = ((uint32_t)e << 10) | (man >> 13);
    const uint32_t rem = man & 0x1FFFu;
    if (rem > 0x1000u || (rem == 0x1000u && (out & 1u))) ++out;
    return sign | (uint16_t)out;
}

__device__ float pack_f16_to_f32(uint16_t h) {
    const uint32_t sign = (uint32_t)(h & 0x8000u) << 16;
    uint32_t ex = (h >> 10) & 0x1Fu, man = h & 0x3FFu;
    if (ex == 0) {
        if (!man) return __builtin_bit_cast(float, sign);
        int sh = 0;
        while (!(man & 0x400u)) {
            man <<= 1;
            ++sh;
        }
        return __builtin_bit_cast(float, sign | ((uint32_t)(113 - sh) << 23) | ((man & 0x3FFu) << 13));
    }
    if (ex == 31) return __builtin_bit_cast(float, sign | 0x7F800000u | (man << 13));
    return __builtin_bit_cast(float, sign | ((ex + 112) << 23) | (man << 13));
}

__device__ __forceinline__ float bf16_bits_to_f32(uint16_t b) { return __builtin_bit_cast(float, (uint32_t)b << 16); }

__device__ __forceinline__ uint16_t scale_of_max(float mx) {  // lib.rs:408-411
    return pack_f32_to_f16(__fdiv_rn(2.0f * (mx == 0.f ? 1.f : mx), 15.0f));
}

// The quantiser word for word (lib.rs:416-427).
__device__ __forceinline__ uint32_t code_exactly(float w, float s) {
    const float q = roundf(__fdiv_rn(w, s));
    long long raw;  // Rust `as i32`: saturating, NaN -> 0
    if (q != q) raw = 0;
    else if (q >= 2147483647.0f) raw = 2147483647LL;
    else if (q <= -2147483648.0f) raw = -2147483648LL;
    else raw = (long long)q;
    long long code = raw + 8;  // an i32 sum in the reference (lib.rs:423): wraps from a saturated raw
    if (code > 2147483647LL) code -= 4294967296LL;
    return (uint32_t)(code < 0 ? 0 : (code > 15 ? 15 : code));
}

// A block of the quantiser covers 128 columns x 128 rows (one group): wavefront t its rows 32 t ... 32 t + 31, lane
// cg + 16 kq the eight columns 8 cg ... of the eight rows 8 kq ..., i.e. eight 16-byte loads a thread, all in flight at
// once, and exactly the rows of one word of each of its columns (layout.h).
constexpr int kQuantCols = 128;
struct QuantTile {
    u32x4 row[8];
    __device__ __forceinline__ void load(const uint16_t *__restrict__ w, int n, int g, int col0, int lane, int t) {
        const uint16_t *src = w + (size_t)(g * kGroupK + 32 * t + 8 * (lane >> 4)) * n + col0 + 8 * (lane & 15);
        if (__builtin_expect((reinterpret_cast<uintptr_t>(w) & 15) == 0, 1)) {
#pragma unroll
            for (int j = 0; j < 8; ++j) row[j] = *reinterpret_cast<const u32x4 *>(src + (size_t)j * n);
        } else {  // a weight that starts off the 16-byte grid
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    row[j][i] = src[(size_t)j * n + 2 * i] | ((uint32_t)src[(size_t)j * n + 2 * i + 1] << 16);
        }
    }
    __device__ __forceinline__ bool all_finite() const {  // no half at or above 0x7F80
        const u32x4 m = fold([](uint32_t v) { return v & 0x7FFF7FFFu; });
        uint32_t over = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) over |= (m[i] + 0x00800080u) & 0x80008000u;
        return over == 0;
    }
    // bits of max |w| of the lane's column pairs over its eight rows; a NaN counts as 0, as in the host's
    // std::max(acc, fabs(w)), which keeps acc where w is NaN
    __device__ __forceinline__ u32x4 max_bits() const {
        u32x4 m = fold([](uint32_t v) { return v & 0x7FFF7FFFu; });
        uint32_t nan = 0;  // a half above 0x7F80 (infinity) carries into its sign bit
#pragma unroll
        for (int i = 0; i < 4; ++i) nan |= (m[i] + 0x007F007Fu) & 0x80008000u;
        if (nan) m = fold([](uint32_t v) {
            v &= 0x7FFF7FFFu;
            return ((v & 0xFFFFu) > 0x7F80u ? 0u : v & 0xFFFFu) | ((v >> 16) > 0x7F80u ? 0u : v & 0xFFFF0000u);
        });
        return m;
    }
    template <class F>
    __device__ __forceinline__ u32x4 fold(F f) const {
        u32x4 m;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            m[i] = f(row[0][i]);
#pragma unroll
            for (int j = 1; j < 8; ++j) m[i] = max_pair(m[i], f(row[j][i]));
        }
        return m;
    }
    static __device__ __forceinline__ uint32_t max_pair(uint32_t a, uint32_t b) {  // v_pk_max_u16
        typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
    }
};

// Column maxima of one group's 128 columns, in LDS as bf16 pairs [wavefront][cg]; a barrier makes them readable.
__device__ __forceinline__ void meet_maxima(u32x4 m, int lane, int t, u32x4 (*part)[16]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        m[i] = QuantTile::max_pair(m[i], (uint32_t)__shfl_xor((int)m[i], 16));
        m[i] = QuantTile::max_pair(m[i], (uint32_t)__shfl_xor((int)m[i], 32));
    }
    if (lane < 16) part[t][lane] = m;
}
__device__ __forceinline__ uint32_t column_max_bits(const u32x4 (*part)[16], int col) {
    const uint16_t *p = reinterpret_cast<const uint16_t *>(part);
    uint32_t m = 0;
#pragma unroll
    for (int t = 0; t < 4; ++t) m = max(m, (uint32_t)p[t * kQuantCols + col]);
    return m;
}

// The weights of one launch: a grid of its own for each, one behind the other, 128 columns by 128 rows a block and
// the columns first; gate and up go into their interleaved pack as well, instead of through a copy of both packed forms.
// Bound by memory: a layer of seven weights (2560 wide, 9216 inside), 107 M in all, 214 MB read and 81 MB written,
// 51 us, 5.8 TB/s (in a launch per weight and a copy 79 us; the load call 145 -> 98).
constexpr int kQuantMany = 16;
constexpr uint32_t kQuantMostBlocks = 1u << 23;
struct QuantMany {
    struct Item {
        const uint16_t *w;
        uint16_t *scales;
        u32x4 *b;
        u32x4 *pair_b;  // null, or the interleaved pack of gate and up that the weight is half of
        uint16_t *pair_s;
        int n, G, pair_side, pad;
    };
    uint32_t end[kQuantMany];  // the first block past each weight's; past the last weight: the largest number
    Item item[kQuantMany];
};
// The block's weight, column and group.
__device__ __forceinline__ const QuantMany::Item &quant_block(const QuantMany &many, int *col0, int *g) {
    int i = 0;
    uint32_t first = 0;
#pragma unroll
    for (int j = 0; j < kQuantMany - 1; ++j)
        if (blockIdx.x >= many.end[j]) {
            i = j + 1;
            first = many.end[j];
        }
    const QuantMany::Item &it = many.item[i];
    const uint32_t columns = (uint32_t)it.n / kQuantCols, block = blockIdx.x - first;
    *g = (int)(block / columns);
    *col0 = (int)(block - (uint32_t)*g * columns) * kQuantCols;
    return it;
}

// One scale for all of K: first the maxima of every group, [G][n] bf16 bits (they lie where the words will) ...
__global__ __launch_bounds__(256) void w4a16_pack_group_max_kernel(const QuantMany many) {
    __shared__ u32x4 part[4][16];
    int col0, g;
    const QuantMany::Item &it = quant_block(many, &col0, &g);
    const int lane = threadIdx.x & 63, t = threadIdx.x >> 6, n = it.n;
    uint16_t *const group_max = reinterpret_cast<uint16_t *>(it.b);
    QuantTile tile;
    tile.load(it.w, n, g, col0, lane, t);
    meet_maxima(tile.max_bits(), lane, t, part);
    __syncthreads();
    if (threadIdx.x < kQuantCols) group_max[(size_t)g * n + col0 + threadIdx.x] = (uint16_t)column_max_bits(part, threadIdx.x);
}
// ... then theirs: block = 64 columns x 4 lanes over the groups.  A few microseconds whatever the weight, so those of a call are
// one launch (seven weights of a layer, 2560 / 9216 wide: the load call 172 -> 140 us, 1280 / 4096 wide 111 -> 68).
__global__ __launch_bounds__(256) void w4a16_pack_column_scale_kernel(const QuantMany many) {
    __shared__ uint32_t part[4][64];
    int i = 0;
    uint32_t block = blockIdx.x;
#pragma unroll
    for (int j = 0; j < kQuantMany - 1; ++j) {
        const uint32_t pieces = (uint32_t)many.item[j].n / 64;
        if (i == j && block >= pieces) {
            block -= pieces;
            i = j + 1;
        }
    }
    const QuantMany::Item &it = many.item[i];
    const int n = it.n, G = it.G;
    const uint16_t *__restrict__ const group_max = reinterpret_cast<const uint16_t *>(it.b);
    const int c = threadIdx.x & 63, gl = threadIdx.x >> 6, col = (int)block * 64 + c;
    uint32_t m = 0;
#pragma unroll 4
    for (int g = gl; g < G; g += 4) m = max(m, (uint32_t)group_max[(size_t)g * n + col]);
    part[gl][c] = m;
    __syncthreads();
    if (gl != 0) return;
#pragma unroll
    for (int i = 1; i < 4; ++i) m = max(m, part[i][c]);
    it.scales[scale_index(0, col, 1)] = scale_of_max(bf16_bits_to_f32((uint16_t)m));
}

// Quantise and pack, the weight read once (it is held in registers between the maxima and the codes; as a kernel
// for the scales and one for the codes with 2-byte loads the same work ran at 1.4 TB/s: 2560 x 9216 34 + 39 us).
// GROUP_SCALES: form the group's scales and write them; else they are there.
//
// Codes by multiplication, the same integers as roundf(fl(w / s)): w has 8 significant bits and s 11, so for a half
// h <= 8.5 (beyond, the code is 0 or 15 whatever the digits) h * s has 16 and w / s is either h itself or at least
// 2^-15 of h away from it.  y = w * rcp(s) * (1 + 2^-19) is within 2^-18 of w / s, relatively: it lies past every half that
// w / s reaches, ties among them, and short of every other, so its nearest integer is w / s rounded with ties
// away from zero.  (Ties are common -- 2 max / 15 is often exact in fp16, then max / s = 7.5 -- so they cannot be left
// to a slow path.)  Only where a weight is not finite or the scale is zero are codes formed step by step.  An IEEE
// division per weight would be 110 us of vector work for the 107 M weights of a layer that take 43 us to read.
template <bool GROUP_SCALES>
__global__ __launch_bounds__(256) void w4a16_pack_quantise_kernel(const QuantMany many) {
    __shared__ u32x4 part[4][16];
    __shared__ __attribute__((aligned(16))) float s_col[kQuantCols], r_col[kQuantCols];
    constexpr int kLanePad = 68, kTilePad = 4 * kLanePad;  // words per 16 lanes / per column tile: 64 and 256, padded against bank conflicts
    __shared__ __attribute__((aligned(16))) uint32_t words[8 * kTilePad];
    int col0, g;
    const QuantMany::Item &it = quant_block(many, &col0, &g);
    const uint16_t *__restrict__ w = it.w;
    uint16_t *__restrict__ scales = it.scales;
    const int n = it.n, G = it.G, pair_side = it.pair_side;
    const int lane = threadIdx.x & 63, t = threadIdx.x >> 6;
    const int cg = lane & 15, kq = lane >> 4;
    QuantTile tile;
    tile.load(w, n, g, col0, lane, t);
    const bool finite = tile.all_finite();
    if constexpr (GROUP_SCALES) {
        meet_maxima(tile.max_bits(), lane, t, part);
        __syncthreads();
    }
    if (threadIdx.x < kQuantCols) {
        const size_t si = scale_index(GROUP_SCALES ? g : 0, col0 + threadIdx.x, GROUP_SCALES ? G : 1);
        uint16_t bits;
        if constexpr (GROUP_SCALES) {
            bits = scale_of_max(bf16_bits_to_f32((uint16_t)column_max_bits(part, threadIdx.x)));
            scales[si] = bits;
        } else {
            bits = scales[si];
        }
        if (it.pair_b && (GROUP_SCALES || g == 0)) {
            const int j = (col0 + threadIdx.x) >> 3;
            it.pair_s[scale_index(g, j * kTileN + 8 * pair_side + (threadIdx.x & 7), GROUP_SCALES ? G : 1)] = bits;
        }
        const float s = pack_f16_to_f32(bits);
        s_col[threadIdx.x] = s;
        r_col[threadIdx.x] = __builtin_amdgcn_rcpf(s) * (1.f + 0x1p-19f);
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const float r = r_col[8 * cg + c];
        uint32_t word = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            // byte b of the word: rows j, j + 2 (nibble_pos), the first in its low nibble
            float v[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint32_t pair = tile.row[4 * (b & 1) + (b >> 1) + 2 * i][c >> 1];
                const float x = __builtin_bit_cast(float, (c & 1) ? pair & 0xFFFF0000u : pair << 16);
                v[i] = __builtin_amdgcn_fmed3f(__builtin_rintf(x * r), -8.f, 7.f);
            }
            word = (uint32_t)__builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(v[1], 16.f, v[0]) + 136.f, b, word);
        }
        if (__builtin_expect(!finite || r == __builtin_inff(), 0)) {
            const uint16_t *src = w + (size_t)(g * kGroupK + 32 * t + 8 * kq) * n + col0 + 8 * cg + c;
            const float s = s_col[8 * cg + c];
            word = 0;
#pragma unroll 1
            for (int j = 0; j < 8; ++j) word |= code_exactly(bf16_bits_to_f32(src[(size_t)j * n]), s) << (4 * nibble_pos(j));
        }
        words[(cg >> 1) * kTilePad + kq * kLanePad + ((cg & 1) * 8 + c) * 4 + t] = word;
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int u = p * 256 + threadIdx.x, nt = u >> 6, l = u & 63;  // chunk lane l of column tile nt
        const u32x4 v = *reinterpret_cast<const u32x4 *>(words + nt * kTilePad + (l >> 4) * kLanePad + (l & 15) * 4);
        it.b[((size_t)(col0 / kTileN + nt) * G + g) * (kChunkWords / 4) + l] = v;
        // columns 8 j ... + 7 are the first half (gate) or the second (up) of tile j of the pair
        if (it.pair_b) {
            const int j = 2 * (col0 / kTileN + nt) + ((l >> 3) & 1);
            it.pair_b[((size_t)j * G + g) * (kChunkWords / 4) + (l & ~15) + 8 * pair_side + (l & 7)] = v;
        }
    }
}

// Gate and up of equal shape into the pack the fused SwiGLU entry point reads (output tile j = gate
// columns 8 j ... 8 j + 7, then the same up columns: kiln_w4a16_interleave_gate_up on the host).  One
// wavefront per output chunk: lane c + 16 kq copies the 16 bytes of its source lane.
__global__ __launch_bounds__(256) void w4a16_interleave_kernel(const u32x4 *__restrict__ gate_b,
                                                               const uint16_t *__restrict__ gate_s,
                                                               const u32x4 *__restrict__ up_b,
                                                               const uint16_t *__restrict__ up_s, int G, int Gs,
                                                               u32x4 *__restrict__ out_b, uint16_t *__restrict__ out_s) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j = blockIdx.x * 4 + wave, g = blockIdx.y;
    const int c = lane & 15, kq = lane >> 4;
    const int src_tile = j >> 1, src_c = 8 * (j & 1) + (c & 7);
    const bool up = (c & 8) != 0;
    const u32x4 *src_b = up ? up_b : gate_b;
    out_b[((size_t)j * G + g) * (kChunkWords / 4) + lane] = src_b[((size_t)src_tile * G + g) * (kChunkWords / 4) + src_c + 16 * kq];
    if (g < Gs && kq == 0) {
        const uint16_t *src_s = up ? up_s : gate_s;
        out_s[((size_t)j * Gs + g) * kTileN + c] = src_s[((size_t)src_tile * Gs + g) * kTileN + src_c];
    }
}

// GPTQ-canonical tensors (qweight [k/8, n] int32 with row j of eight in bits 4 j, scales [k/g, n] fp16;
// crates/kiln-model/src/quantized.rs:1-14, :127-152) into the tile layout: kiln_w4a16_repack_gptq on the
// host.  One wavefront per chunk; lane c + 16 kq gathers its four source words and moves each nibble to
// its place in the layout's word.  No re-quantisation: the codes are the checkpoint's.
__device__ __forceinline__ uint32_t pack_shuffle_nibbles(uint32_t w) {
    uint32_t out = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) out |= ((w >> (4 * j)) & 0xFu) << (4 * nibble_pos(j));
    return out;
}

__global__ __launch_bounds__(256) void w4a16_repack_gptq_kernel(const uint32_t *__restrict__ qweight,
                                                                const uint16_t *__restrict__ scales, int n, int G, int Gs,
                                                                u32x4 *__restrict__ b_packed,
                                                                uint16_t *__restrict__ scales_tiled) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nt = blockIdx.x * 4 + wave, g = blockIdx.y;
    const int c = lane & 15, kq = lane >> 4;
    const int col = nt * kTileN + c;
    uint32_t words[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
        words[t] = pack_shuffle_nibbles(qweight[(size_t)((g * kGroupK + 32 * t + 8 * kq) / 8) * n + col]);
    b_packed[((size_t)nt * G + g) * (kChunkWords / 4) + lane] = u32x4{words[0], words[1], words[2], words[3]};
    if (g < Gs && kq == 0) scales_tiled[scale_index(g, col, Gs)] = scales[(size_t)g * n + col];
}

// 1 in *bad if any packed zero-point word differs from 0x88888888 (zero-point 8 in all eight nibbles)
__global__ void w4a16_check_qzeros_kernel(const uint32_t *__restrict__ qzeros, size_t count, int *bad) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x)
        if (qzeros[i] != 0x88888888u) *bad = 1;
}
__global__ void w4a16_clear_flag_kernel(int *flag) { *flag = 0; }

}  // namespace
}  // namespace kiln

extern "C" kiln_marlin_status_t kiln_w4a16_repack_gptq_device(const void *qweight, const void *scales, const void *qzeros,
                                                              int k, int n, int groupsize, void *b_packed,
                                                              void *scales_tiled, int dev, void *stream) {
    using namespace kiln;
    (void)dev;
    if (!qweight || !scales || !b_packed || !scales_tiled) return KILN_W4A16_ERR_ARGUMENT;
    if (k <= 0 || n <= 0 || k % 128 != 0 || n % 256 != 0 || !(groupsize == -1 || groupsize == 128))
        return KILN_W4A16_ERR_PROB_SHAPE;
    const int G = k / kGroupK, Gs = groupsize == -1 ? 1 : G;
    if (G > 65535) return KILN_W4A16_ERR_PROB_SHAPE;  // grid y
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (qzeros) {
        // the zero-points must all be 8, as on the host route; the answer is needed before anything is written, so
        // this one check waits for the stream.  The flag lives at the start of the output and is overwritten below.
        int *flag = reinterpret_cast<int *>(b_packed);
        int bad = 0;
        w4a16_clear_flag_kernel<<<1, 1, 0, st>>>(flag);
        w4a16_check_qzeros_kernel<<<64, 256, 0, st>>>((const uint32_t *)qzeros, (size_t)Gs * (n / 8), flag);
        if (hipGetLastError() != hipSuccess ||
            hipMemcpyAsync(&bad, flag, sizeof(int), hipMemcpyDeviceToHost, st) != hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess)
            return KILN_W4A16_ERR_LAUNCH;
        if (bad) return KILN_W4A16_ERR_ZERO_POINT;
    }
    w4a16_repack_gptq_kernel<<<dim3(n / 64, G), 256, 0, st>>>((const uint32_t *)qweight, (const uint16_t *)scales, n, G, Gs,
                                                               (u32x4 *)b_packed, (uint16_t *)scales_tiled);
    return hipGetLastError() == hipSuccess ? KILN_W4A16_OK : KILN_W4A16_ERR_LAUNCH;
}

extern "C" kiln_marlin_status_t kiln_w4a16_interleave_gate_up_device(const void *gate_b, const void *gate_s,
                                                                     const void *up_b, const void *up_s, int k,
                                                                     int n_each, int groupsize, void *out_b,
                                                                     void *out_s, int dev, void *stream) {
    using namespace kiln;
    (void)dev;
    if (!gate_b || !gate_s || !up_b || !up_s || !out_b || !out_s) return KILN_W4A16_ERR_ARGUMENT;
    if (k <= 0 || k % 128 != 0 || n_each <= 0 || n_each % 128 != 0 || !(groupsize == -1 || groupsize == 128))
        return KILN_W4A16_ERR_PROB_SHAPE;
    const int G = k / kGroupK, Gs = groupsize == -1 ? 1 : G;
    if (G > 65535) return KILN_W4A16_ERR_PROB_SHAPE;  // grid y
    w4a16_interleave_kernel<<<dim3(n_each / 8 / 4, G), 256, 0, reinterpret_cast<hipStream_t>(stream)>>>(
        (const u32x4 *)gate_b, (const uint16_t *)gate_s, (const u32x4 *)up_b, (const uint16_t *)up_s, G, Gs,
        (u32x4 *)out_b, (uint16_t *)out_s);
    return hipGetLastError() == hipSuccess ? KILN_W4A16_OK : KILN_W4A16_ERR_LAUNCH;
}

extern "C" kiln_marlin_status_t kiln_w4a16_quantize_and_pack_many_device(const kiln_w4a16_quantize_item *items, int count, int dev,
                                                                         void *stream) {
    using namespace kiln;
    (void)dev;
    if (count < 0 || (count > 0 && !items)) return KILN_W4A16_ERR_ARGUMENT;
    for (int i = 0; i < count; ++i) {
        const kiln_w4a16_quantize_item &q = items[i];
        if (q.k <= 0 || q.n <= 0 || q.k % 128 != 0 || q.n % 256 != 0 || !(q.groupsize == -1 || q.groupsize == 128))
            return KILN_W4A16_ERR_PROB_SHAPE;
        if (!q.weight_bf16 || !q.b_packed || !q.scales_f16 || !q.pair_b != !q.pair_s || (q.pair_b && (q.pair_side | 1) != 1))
            return KILN_W4A16_ERR_ARGUMENT;
        // (2^23 blocks are a weight of 256 GiB; a launch takes fewer than 2^24)
        if (q.k / kGroupK > 65535 || (uint64_t)(q.n / kQuantCols) * (q.k / kGroupK) > kQuantMostBlocks) return KILN_W4A16_ERR_PROB_SHAPE;
    }
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    for (const int groupsize : {128, -1}) {
        for (int i = 0; i < count;) {
            QuantMany many = {};
            int here = 0;
            uint32_t blocks = 0;
            // as many as fit one launch, by number and by blocks
            for (; i < count && here < kQuantMany; ++i) {
                const kiln_w4a16_quantize_item &q = items[i];
                if (q.groupsize != groupsize) continue;
                const uint32_t more = (uint32_t)(q.n / kQuantCols) * (q.k / kGroupK);
                if (blocks + more > kQuantMostBlocks) break;
                blocks += more;
                many.end[here] = blocks;
                many.item[here++] = {(const uint16_t *)q.weight_bf16, (uint16_t *)q.scales_f16, (u32x4 *)q.b_packed, (u32x4 *)q.pair_b,
                                     (uint16_t *)q.pair_s, q.n, q.k / kGroupK, q.pair_side, 0};
            }
            if (here == 0) break;
            for (int j = here; j < kQuantMany; ++j) many.end[j] = 0xFFFFFFFFu;
            if (groupsize == 128) {
                w4a16_pack_quantise_kernel<true><<<blocks, 256, 0, st>>>(many);
            } else {
                w4a16_pack_group_max_kernel<<<blocks, 256, 0, st>>>(many);
                uint32_t pieces = 0;
                for (int j = 0; j < here; ++j) pieces += (uint32_t)many.item[j].n / 64;
                w4a16_pack_column_scale_kernel<<<pieces, 256, 0, st>>>(many);
                w4a16_pack_quantise_kernel<false><<<blocks, 256, 0, st>>>(many);
            }
        }
    }
    return hipGetLastError() == hipSuccess ? KILN_W4A16_OK : KILN_W4A16_ERR_LAUNCH;
}

extern "C" kiln_marlin_status_t kiln_w4a16_quantize_and_pack_device(const void *weight_bf16, int k, int n, int groupsize,
                                                                    void *b_packed, void *scales_f16, int dev,
                                                                    void *stream) {
    const kiln_w4a16_quantize_item item = {weight_bf16, k, n, groupsize, 0, b_packed, scales_f16, nullptr, nullptr};
    return kiln_w4a16_quantize_and_pack_many_device(&item, 1, dev, stream);
}
