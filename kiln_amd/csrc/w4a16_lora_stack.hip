// The adapters of projections that run as one GEMM (side by side, or gate and up interleaved) as one stacked
// set: A row-concatenated, B block-structured, the stacked rank rounded up to a multiple of 8 with zeros.
// What crates/kiln-model/src/adapter_merge.rs:639-712 does once per merge, for adapters that arrive per call.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kiln_w4a16.h"
#include "device_common.h"

namespace kiln {
namespace {

constexpr int kMaxStackBlocks = 8;

struct StackBlocks {
    const uint16_t *a[kMaxStackBlocks];  // bf16 [rank, K]
    const uint16_t *b[kMaxStackBlocks];  // bf16 [rows, rank]
    int col[kMaxStackBlocks + 1];        // first column on the stacked rank axis; [count] = their sum
    int first[kMaxStackBlocks];          // first row of the GEMM's B (interleaved: 0 = gate's rows, 8 = up's)
    int rows[kMaxStackBlocks];
    int count;
};

// One 16-byte unit of either result per thread: units of A first, then those of B.  Bound by the launch (245 KB of
// A and 1 MB of B for q | k | v with rank 16 each: 3 us), and in one launch where torch needs four to eight.
__global__ __launch_bounds__(256) void w4a16_lora_stack_kernel(StackBlocks s, int K, int N, int r_total, int interleaved,
                                                               u32x4 *__restrict__ a_cat, u32x4 *__restrict__ b_cat) {
    const int a_units = r_total * (K / 8), b_units = N * (r_total / 8);
    int u = blockIdx.x * 256 + threadIdx.x;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (u < a_units) {
        const int row = u / (K / 8), k8 = u - row * (K / 8);
#pragma unroll
        for (int i = 0; i < kMaxStackBlocks; ++i)
            if (i < s.count && row >= s.col[i] && row < s.col[i + 1])
                v = *reinterpret_cast<const u32x4 *>(s.a[i] + (size_t)(row - s.col[i]) * K + k8 * 8);
        a_cat[u] = v;
        return;
    }
    u -= a_units;
    if (u >= b_units) return;
    const int row = u / (r_total / 8), c0 = (u - row * (r_total / 8)) * 8;
#pragma unroll
    for (int i = 0; i < kMaxStackBlocks; ++i) {
        if (i >= s.count) break;
        const int r = interleaved ? (row >> 4) * 8 + (row & 7) : row - s.first[i];
        if (interleaved ? (row & 8) != s.first[i] : (r < 0 || r >= s.rows[i])) continue;
        const int lo = s.col[i], rank = s.col[i + 1] - lo;
        const uint16_t *src = s.b[i] + (size_t)r * rank;
        if (((lo | rank) & 7) == 0) {  // whole units
            if (c0 >= lo && c0 < lo + rank) v = *reinterpret_cast<const u32x4 *>(src + (c0 - lo));
        } else {
            uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (c0 + j >= lo && c0 + j < lo + rank) w[j >> 1] |= (uint32_t)src[c0 + j - lo] << (16 * (j & 1));
            v = u32x4{w[0], w[1], w[2], w[3]};
        }
    }
    b_cat[u] = v;
}

}  // namespace
}  // namespace kiln

extern "C" kiln_marlin_status_t kiln_w4a16_stack_adapters(const void *const *lora_a, const void *const *lora_b,
                                                          const int *ranks, const int *first_rows, const int *rows,
                                                          int count, int prob_k, int prob_n, int r_total, int interleaved,
                                                          void *a_cat, void *b_cat, void *stream) {
    using namespace kiln;
    if (!lora_a || !lora_b || !ranks || !first_rows || !rows || !a_cat || !b_cat) return KILN_W4A16_ERR_ARGUMENT;
    if (count < 1 || count > kMaxStackBlocks || r_total < 1 || r_total > 64 || r_total % 8 != 0) return KILN_W4A16_ERR_KERN_SHAPE;
    if (prob_k <= 0 || prob_k % 128 != 0 || prob_n <= 0 || prob_n % 256 != 0 || prob_n > INT32_MAX / 8 || prob_k > INT32_MAX / 8)
        return KILN_W4A16_ERR_PROB_SHAPE;
    StackBlocks s{};
    s.count = count;
    int col = 0;
    for (int i = 0; i < count; ++i) {
        // every address the kernel forms lies inside a block's own [rank, K] and [rows, rank]
        if (!lora_a[i] || !lora_b[i] || ranks[i] < 1 || col + ranks[i] > r_total) return KILN_W4A16_ERR_ARGUMENT;
        if (interleaved ? (rows[i] != prob_n / 2 || (first_rows[i] != 0 && first_rows[i] != 8))
                        : (first_rows[i] < 0 || rows[i] < 1 || rows[i] > prob_n - first_rows[i]))
            return KILN_W4A16_ERR_ARGUMENT;
        for (const void *p : {lora_a[i], lora_b[i]})
            if (reinterpret_cast<uintptr_t>(p) % 16 != 0) return KILN_W4A16_ERR_ARGUMENT;
        s.a[i] = (const uint16_t *)lora_a[i];
        s.b[i] = (const uint16_t *)lora_b[i];
        s.first[i] = first_rows[i];
        s.rows[i] = rows[i];
        s.col[i] = col;
        col += ranks[i];
        s.col[i + 1] = col;
    }
    const int units = r_total * (prob_k / 8) + prob_n * (r_total / 8);
    w4a16_lora_stack_kernel<<<(units + 255) / 256, 256, 0, reinterpret_cast<hipStream_t>(stream)>>>(
        s, prob_k, prob_n, r_total, interleaved ? 1 : 0, (u32x4 *)a_cat, (u32x4 *)b_cat);
    return hipGetLastError() == hipSuccess ? KILN_W4A16_OK : KILN_W4A16_ERR_LAUNCH;
}
