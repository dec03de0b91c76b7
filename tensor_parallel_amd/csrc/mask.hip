// The causal attention mask of a forward on a static cache: out[i][j] = (kv_offset + j <= *q_offset + i), one byte each.
//
// Latency-bound (a decode step's mask is one row of a few thousand bytes): what counts is that it is one launch. Built from torch
// calls it is seven (four ranges, two additions, the comparison), two to four microseconds each in a recorded step, once per rank.
// Two-layer Llama-shaped decoder of two ranks, recorded step: one row on 500 positions 347 -> 327 us, 8 on 2048 510 -> 483, 40 on 1000 572 -> 539.
#include "common.h"

namespace tpamd {
namespace {

__global__ __launch_bounds__(256) void causal_mask_kernel(const int64_t *q_offset, int64_t kv_offset, int64_t rows, int64_t cols, uint8_t *out) {
    const int64_t j = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (j >= cols) return;
    const int64_t first = *q_offset;
    for (int64_t i = blockIdx.y; i < rows; i += gridDim.y) out[i * cols + j] = kv_offset + j <= first + i ? 1 : 0;
}

}  // namespace
}  // namespace tpamd

using namespace tpamd;

extern "C" int tpamd_causal_mask(const int64_t *q_offset_dev, int64_t kv_offset, int64_t rows, int64_t cols, void *mask_dev, void *stream) {
    const char *who = "tpamd_causal_mask";
    TPAMD_REQUIRE(rows >= 0 && cols >= 0 && cols < (1ll << 31) && rows < (1ll << 31), "%s: bad dimension", who);
    if (rows == 0 || cols == 0) return TPAMD_OK;
    TPAMD_REQUIRE(q_offset_dev && mask_dev, "%s: null pointer", who);
    const dim3 grid(static_cast<unsigned>((cols + 255) / 256), static_cast<unsigned>(rows < 65535 ? rows : 65535));
    hipLaunchKernelGGL(causal_mask_kernel, grid, dim3(256), 0, static_cast<hipStream_t>(stream), q_offset_dev, kv_offset, rows, cols,
                       static_cast<uint8_t *>(mask_dev));
    TPAMD_HIP(hipGetLastError());
    return TPAMD_OK;
}
