// The causal attention mask of a forward on a static cache: out[i][j] = (kv_offset + j <= *q_offset + i), one byte each.
//
// Latency-bound (a decode step's mask is one row of a few thousand bytes): what counts is that it is one launch. Built from torch
// calls it is seven (four ranges, two additions, the comparison), two to four microseconds each in a recorded step, once per rank.
// Two-layer Llama-shaped decoder of two ranks, recorded step: one row on 500 positions 347 -> 327 us, 8 on 2048 510 -> 483, 40 on 1000 572 -> 539.
#include "common.h"

namespace tpamd {
namespace {

// blockIdx.z = 1: the mask of a second rank, byte distances to its operands.
__global__ __launch_bounds__(256) void causal_mask_kernel(const int64_t *q_offset, int64_t kv_offset, int64_t rows, int64_t cols, uint8_t *out, int64_t to_offset,
                                                          int64_t to_out) {
    const int64_t j = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (j >= cols) return;
    if (blockIdx.z != 0) {
        q_offset = reinterpret_cast<const int64_t *>(reinterpret_cast<const char *>(q_offset) + to_offset);
        out += to_out;
    }
    const int64_t first = *q_offset;
    for (int64_t i = blockIdx.y; i < rows; i += gridDim.y) out[i * cols + j] = kv_offset + j <= first + i ? 1 : 0;
}

// The counts of cached positions of several ranks, advanced by one launch of one wavefront: latency, 4.5 us in a recorded step and layer where torch's
// additions took 1.9-4.6 us for each of two ranks (with the additions behind the MLPs, the tables and the mask of both ranks in one launch each:
// 260 -> 249 us of a two-layer step of one row, 408 -> 400 of 40).
struct Counts {
    int64_t *at[8];
};
__global__ __launch_bounds__(64) void advance_kernel(Counts counts, int n, int64_t by) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if (i < n && static_cast<int>(threadIdx.x) == i) *counts.at[i] += by;
}

}  // namespace
}  // namespace tpamd

using namespace tpamd;

extern "C" int tpamd_causal_mask(const int64_t *q_offset_dev, int64_t kv_offset, int64_t rows, int64_t cols, void *mask_dev, void *stream) {
    const void *offset = q_offset_dev;
    return tpamd_causal_mask_ranks(1, &offset, kv_offset, rows, cols, &mask_dev, stream);
}

extern "C" int tpamd_causal_mask_ranks(int n, const void *const *q_offset_dev, int64_t kv_offset, int64_t rows, int64_t cols, void *const *mask_dev, void *stream) {
    const char *who = "tpamd_causal_mask";
    TPAMD_REQUIRE(n >= 0 && q_offset_dev && mask_dev, "%s: null pointer", who);
    TPAMD_REQUIRE(rows >= 0 && cols >= 0 && cols < (1ll << 31) && rows < (1ll << 31), "%s: bad dimension", who);
    if (rows == 0 || cols == 0) return TPAMD_OK;
    for (int i = 0; i < n; ++i) TPAMD_REQUIRE(q_offset_dev[i] && mask_dev[i], "%s: null pointer", who);
    // grids of fewer than 2^32 threads: rows beyond those of a grid are taken by its blocks in turn
    const int64_t blocks = (cols + 255) / 256, most = ((1ll << 23) - 1) / blocks > 0 ? ((1ll << 23) - 1) / blocks : 1;
    const int64_t height = rows < most ? rows : most;
    const int together = blocks < (1 << 22) ? 2 : 1;
    for (int i = 0; i < n; i += together) {
        const bool two = together == 2 && i + 1 < n;
        const dim3 grid(static_cast<unsigned>(blocks), static_cast<unsigned>(height < 65535 ? height : 65535), two ? 2 : 1);
        hipLaunchKernelGGL(causal_mask_kernel, grid, dim3(256), 0, static_cast<hipStream_t>(stream), static_cast<const int64_t *>(q_offset_dev[i]), kv_offset, rows, cols,
                           static_cast<uint8_t *>(mask_dev[i]), two ? bytes_from(q_offset_dev[i], q_offset_dev[i + 1]) : 0,
                           two ? bytes_from(mask_dev[i], mask_dev[i + 1]) : 0);
    }
    TPAMD_HIP(hipGetLastError());
    return TPAMD_OK;
}

extern "C" int tpamd_advance_ranks(int n, void *const *counts_dev, int64_t by, void *stream) {
    const char *who = "tpamd_advance_ranks";
    TPAMD_REQUIRE(n >= 0 && counts_dev, "%s: null pointer", who);
    for (int i = 0; i < n; i += 8) {
        Counts counts{};
        const int part = n - i < 8 ? n - i : 8;
        for (int j = 0; j < part; ++j) {
            TPAMD_REQUIRE(counts_dev[i + j] && aligned(counts_dev[i + j], 8), "%s: a count must be an aligned int64", who);
            counts.at[j] = static_cast<int64_t *>(counts_dev[i + j]);
        }
        hipLaunchKernelGGL(advance_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream), counts, part, by);
    }
    TPAMD_HIP(hipGetLastError());
    return TPAMD_OK;
}
