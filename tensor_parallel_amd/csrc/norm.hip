// RMS normalisation of the rows of an activation, in one pass: y = w * round(x * rsqrt(mean(x^2) + eps)).
//
// Bound: at decode (a few rows) by the latency of one launch, at prefill by HBM (x read once, y written once). The module's
// own forward is eight elementwise and reduction launches on an fp32 copy of x. Ten norms of 4096 elements (a two-layer decoder
// of two ranks): the recorded decode step on one row 530 -> 384 us, the prefill of 4096 rows 4.46 -> 3.51 ms (105 -> 10 us a norm).
//
// A block owns one row and holds it in registers between the two uses (16 bytes per lane and chunk), so that x is read
// once; the partial sums meet in the wavefront's lanes first, then in LDS. Rounding follows the module's own sequence:
// sum and scaling in fp32, the scaled value rounded to the tensor dtype, the product with the weight rounded again.
//
// ADD: x is first added to a second activation r (rounded, and stored as the new residual stream), so that the addition in front of a
// decoder layer's second norm is no launch and no pass of its own: recorded decode step of a two-layer decoder on 8 x 2048 positions 485 -> 477 us, prefill of 4096
// rows 3.42 -> 3.30 ms.
#include "common.h"

namespace tpamd {
namespace {

struct NormParams {
    const char *x, *w, *r;  // r: the addend's rows; layer norm: its bias, or NULL
    char *y, *s;
    int64_t ldx, ldr, ldy;  // elements between rows (ldy: of y and s)
    int D;
    float eps;
    // blockIdx.y = 1: the rows of a second rank, byte distances to its operands (one row of 4096: two launches of 3.1 us, one of 3.7)
    struct { int64_t x, w, r, y, s; } to;
};

__device__ __forceinline__ void take_rank(NormParams &p) {
    if (blockIdx.y == 0) return;
    p.x += p.to.x; p.w += p.to.w; p.r += p.to.r; p.y += p.to.y; p.s += p.to.s;
}

// Sum over the block, the same value in every thread. `part` has one float per wavefront.
template <int WAVES>
__device__ __forceinline__ float block_sum(float v, float *part) {
#pragma unroll
    for (int d = 1; d < 64; d *= 2) v += __shfl_xor(v, d);
    if constexpr (WAVES > 1) {
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
        __syncthreads();
        v = 0.f;
#pragma unroll
        for (int i = 0; i < WAVES; ++i) v += part[i];
    }
    return v;
}

template <int DT>
__device__ __forceinline__ uint32_t scale2(uint32_t x, float r, uint32_t w) {
    const uint32_t n = pack2_half<DT>(lo_half_to_f32<DT>(x) * r, hi_half_to_f32<DT>(x) * r);
    return pack2_half<DT>(lo_half_to_f32<DT>(n) * lo_half_to_f32<DT>(w), hi_half_to_f32<DT>(n) * hi_half_to_f32<DT>(w));
}

template <int DT>
__device__ __forceinline__ uint32_t add2(uint32_t a, uint32_t b) {
    return pack2_half<DT>(lo_half_to_f32<DT>(a) + lo_half_to_f32<DT>(b), hi_half_to_f32<DT>(a) + hi_half_to_f32<DT>(b));
}

// 16-bit rows of D elements, D a multiple of 8 and at most 64 * WAVES * CH * 8, every row on a 16-byte boundary.
template <int DT, int WAVES, int CH, bool ADD>
__global__ __launch_bounds__(64 * WAVES) void rms_norm_kernel(NormParams p) {
    take_rank(p);
    constexpr int T = 64 * WAVES;
    __shared__ float part[WAVES];
    const int64_t row = blockIdx.x;
    const uint4 *x = reinterpret_cast<const uint4 *>(p.x + row * p.ldx * 2);
    const uint4 *w = reinterpret_cast<const uint4 *>(p.w);
    uint4 *y = reinterpret_cast<uint4 *>(p.y + row * p.ldy * 2);
    const int n = p.D / 8;
    uint4 v[CH], wv[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int i = threadIdx.x + c * T;
        v[c] = i < n ? x[i] : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int i = threadIdx.x + c * T;
        wv[c] = i < n ? w[i] : make_uint4(0, 0, 0, 0);
    }
    if constexpr (ADD) {
        const uint4 *r = reinterpret_cast<const uint4 *>(p.r + row * p.ldr * 2);
        uint4 *s = reinterpret_cast<uint4 *>(p.s + row * p.ldy * 2);
        uint4 rv[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int i = threadIdx.x + c * T;
            rv[c] = i < n ? r[i] : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int i = threadIdx.x + c * T;
            v[c] = make_uint4(add2<DT>(rv[c].x, v[c].x), add2<DT>(rv[c].y, v[c].y), add2<DT>(rv[c].z, v[c].z), add2<DT>(rv[c].w, v[c].w));
            if (i < n) s[i] = v[c];
        }
    }
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const uint32_t u[4] = {v[c].x, v[c].y, v[c].z, v[c].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float a = lo_half_to_f32<DT>(u[j]), b = hi_half_to_f32<DT>(u[j]);
            sum = fmaf(a, a, fmaf(b, b, sum));
        }
    }
    const float r = rsqrtf(block_sum<WAVES>(sum, part) / static_cast<float>(p.D) + p.eps);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int i = threadIdx.x + c * T;
        if (i < n)
            y[i] = make_uint4(scale2<DT>(v[c].x, r, wv[c].x), scale2<DT>(v[c].y, r, wv[c].y), scale2<DT>(v[c].z, r, wv[c].z),
                              scale2<DT>(v[c].w, r, wv[c].w));
    }
}

// Any length, alignment and dtype: element loads, x (ADD: the stored sum) read twice (the second time from the cache, by the thread
// that has read or stored it before).
template <int DT, bool ADD>
__global__ __launch_bounds__(256) void rms_norm_any_kernel(NormParams p) {
    take_rank(p);
    __shared__ float part[4];
    const int64_t row = blockIdx.x;
    float sum = 0.f;
    auto load = [](const char *base, int64_t i) {
        if constexpr (DT == TPAMD_F32) return reinterpret_cast<const float *>(base)[i];
        else return half_to_f32<DT>(reinterpret_cast<const uint16_t *>(base)[i]);
    };
    for (int i = threadIdx.x; i < p.D; i += 256) {
        float a = load(p.x, row * p.ldx + i);
        if constexpr (ADD) {
            a += load(p.r, row * p.ldr + i);
            if constexpr (DT == TPAMD_F32) {
                reinterpret_cast<float *>(p.s)[row * p.ldy + i] = a;
            } else {
                const uint16_t h = f32_to_half<DT>(a);
                reinterpret_cast<uint16_t *>(p.s)[row * p.ldy + i] = h;
                a = half_to_f32<DT>(h);
            }
        }
        sum = fmaf(a, a, sum);
    }
    const float r = rsqrtf(block_sum<4>(sum, part) / static_cast<float>(p.D) + p.eps);
    for (int i = threadIdx.x; i < p.D; i += 256) {
        const float n = (ADD ? load(p.s, row * p.ldy + i) : load(p.x, row * p.ldx + i)) * r;
        if constexpr (DT == TPAMD_F32)
            reinterpret_cast<float *>(p.y)[row * p.ldy + i] = n * load(p.w, i);
        else
            reinterpret_cast<uint16_t *>(p.y)[row * p.ldy + i] = f32_to_half<DT>(half_to_f32<DT>(f32_to_half<DT>(n)) * load(p.w, i));
    }
}

// ---- layer norm: y = (x - mean) * rsqrt(var + eps) * w + b, mean and variance of a row in fp32 (two sums over registers, the second of squared
// differences), rounded once, as torch's own. What bounds it is the same as above. torch's kernel gives a row one wavefront: 16 rows of 8192 in
// fp16 took 9.3 us there, rank by rank, and take 4.1 here for two ranks at once; 1024 rows twice 14.4 there and 14.5 for both here.
template <int DT>
struct Chunk {  // 16 bytes
    static constexpr int E = DT == TPAMD_F32 ? 4 : 8;
    float v[E];
};
template <int DT>
__device__ __forceinline__ Chunk<DT> unpack(uint4 u) {
    const uint32_t a[4] = {u.x, u.y, u.z, u.w};
    Chunk<DT> c;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if constexpr (DT == TPAMD_F32) c.v[j] = __uint_as_float(a[j]);
        else {
            c.v[2 * j] = lo_half_to_f32<DT>(a[j]);
            c.v[2 * j + 1] = hi_half_to_f32<DT>(a[j]);
        }
    }
    return c;
}
template <int DT>
__device__ __forceinline__ uint4 pack(const Chunk<DT> &c) {
    uint32_t a[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if constexpr (DT == TPAMD_F32) a[j] = __float_as_uint(c.v[j]);
        else a[j] = pack2_half<DT>(c.v[2 * j], c.v[2 * j + 1]);
    }
    return make_uint4(a[0], a[1], a[2], a[3]);
}

// Rows of D elements in whole 16-byte chunks, at most 64 * WAVES * CH of them, every row, w and b (NULL: none) on a 16-byte boundary.
template <int DT, int WAVES, int CH>
__global__ __launch_bounds__(64 * WAVES) void layer_norm_kernel(NormParams p) {
    take_rank(p);
    constexpr int T = 64 * WAVES, E = Chunk<DT>::E;
    constexpr int64_t ESZ = DT == TPAMD_F32 ? 4 : 2;
    __shared__ float part[2][WAVES];
    const int64_t row = blockIdx.x;
    const uint4 *x = reinterpret_cast<const uint4 *>(p.x + row * p.ldx * ESZ);
    const uint4 *w = reinterpret_cast<const uint4 *>(p.w), *b = reinterpret_cast<const uint4 *>(p.r);
    uint4 *y = reinterpret_cast<uint4 *>(p.y + row * p.ldy * ESZ);
    const int n = p.D / E;
    uint4 raw[CH], wv[CH], bv[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int i = threadIdx.x + c * T;
        raw[c] = i < n ? x[i] : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int i = threadIdx.x + c * T;
        wv[c] = i < n ? w[i] : make_uint4(0, 0, 0, 0);
        bv[c] = i < n && b != nullptr ? b[i] : make_uint4(0, 0, 0, 0);
    }
    Chunk<DT> v[CH];
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        v[c] = unpack<DT>(raw[c]);
#pragma unroll
        for (int e = 0; e < E; ++e) sum += v[c].v[e];
    }
    const float mean = block_sum<WAVES>(sum, part[0]) / static_cast<float>(p.D);
    float sq = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const bool in = static_cast<int>(threadIdx.x) + c * T < n;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            v[c].v[e] -= mean;
            sq = fmaf(in ? v[c].v[e] : 0.f, v[c].v[e], sq);
        }
    }
    const float r = rsqrtf(block_sum<WAVES>(sq, part[1]) / static_cast<float>(p.D) + p.eps);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int i = threadIdx.x + c * T;
        const Chunk<DT> wc = unpack<DT>(wv[c]), bc = unpack<DT>(bv[c]);
#pragma unroll
        for (int e = 0; e < E; ++e) v[c].v[e] = fmaf(v[c].v[e] * r, wc.v[e], bc.v[e]);
        if (i < n) y[i] = pack<DT>(v[c]);
    }
}

// Any length and alignment: element loads, x read three times (from the cache after the first).
template <int DT>
__global__ __launch_bounds__(256) void layer_norm_any_kernel(NormParams p) {
    take_rank(p);
    __shared__ float part[2][4];
    const int64_t row = blockIdx.x;
    auto load = [](const char *base, int64_t i) {
        if constexpr (DT == TPAMD_F32) return reinterpret_cast<const float *>(base)[i];
        else return half_to_f32<DT>(reinterpret_cast<const uint16_t *>(base)[i]);
    };
    float sum = 0.f;
    for (int i = threadIdx.x; i < p.D; i += 256) sum += load(p.x, row * p.ldx + i);
    const float mean = block_sum<4>(sum, part[0]) / static_cast<float>(p.D);
    float sq = 0.f;
    for (int i = threadIdx.x; i < p.D; i += 256) {
        const float d = load(p.x, row * p.ldx + i) - mean;
        sq = fmaf(d, d, sq);
    }
    const float r = rsqrtf(block_sum<4>(sq, part[1]) / static_cast<float>(p.D) + p.eps);
    for (int i = threadIdx.x; i < p.D; i += 256) {
        const float v = fmaf((load(p.x, row * p.ldx + i) - mean) * r, load(p.w, i), p.r != nullptr ? load(p.r, i) : 0.f);
        if constexpr (DT == TPAMD_F32) reinterpret_cast<float *>(p.y)[row * p.ldy + i] = v;
        else reinterpret_cast<uint16_t *>(p.y)[row * p.ldy + i] = f32_to_half<DT>(v);
    }
}

// n: 16-byte chunks per row.
template <int DT>
void launch_layer_rows(const NormParams &p, int64_t rows, int ranks, bool vec, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(rows), ranks);
    const int n = p.D / Chunk<DT>::E;
    if (!vec) hipLaunchKernelGGL((layer_norm_any_kernel<DT>), grid, dim3(256), 0, s, p);
    else if (n <= 64) hipLaunchKernelGGL((layer_norm_kernel<DT, 1, 1>), grid, dim3(64), 0, s, p);
    else if (n <= 256) hipLaunchKernelGGL((layer_norm_kernel<DT, 4, 1>), grid, dim3(256), 0, s, p);
    else if (n <= 512) hipLaunchKernelGGL((layer_norm_kernel<DT, 8, 1>), grid, dim3(512), 0, s, p);
    else if (n <= 1024) hipLaunchKernelGGL((layer_norm_kernel<DT, 8, 2>), grid, dim3(512), 0, s, p);
    else hipLaunchKernelGGL((layer_norm_kernel<DT, 16, 2>), grid, dim3(1024), 0, s, p);
}

template <int DT, bool ADD>
void launch_rows(const NormParams &p, int64_t rows, int ranks, bool vec, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(rows), ranks);
    const int n = p.D / 8;  // 16-byte chunks per row
    // one chunk per lane as far as a block of 16 wavefronts goes: a lone row is then one load away from its sum
    // (4096 elements on 8 wavefronts)
    if (!vec) hipLaunchKernelGGL((rms_norm_any_kernel<DT, ADD>), grid, dim3(256), 0, s, p);
    else if constexpr (DT != TPAMD_F32) {
        if (n <= 64) hipLaunchKernelGGL((rms_norm_kernel<DT, 1, 1, ADD>), grid, dim3(64), 0, s, p);
        else if (n <= 256) hipLaunchKernelGGL((rms_norm_kernel<DT, 4, 1, ADD>), grid, dim3(256), 0, s, p);
        else if (n <= 512) hipLaunchKernelGGL((rms_norm_kernel<DT, 8, 1, ADD>), grid, dim3(512), 0, s, p);
        else if (n <= 1024) hipLaunchKernelGGL((rms_norm_kernel<DT, 8, 2, ADD>), grid, dim3(512), 0, s, p);
        else hipLaunchKernelGGL((rms_norm_kernel<DT, 16, 2, ADD>), grid, dim3(1024), 0, s, p);
    }
}

// A launch has at most 2^32 - 1 threads, and one that asks for more runs, without an error, what is left of the count modulo 2^32: further
// rows go into further launches.
constexpr int64_t ROWS_PER_LAUNCH = 1ll << 20;  // of two ranks, in blocks of up to 1024 threads

template <int DT, bool ADD>
void launch(NormParams p, int64_t rows, int ranks, bool vec, hipStream_t s) {
    constexpr int64_t ESZ = DT == TPAMD_F32 ? 4 : 2;
    for (; rows > 0; rows -= ROWS_PER_LAUNCH) {
        launch_rows<DT, ADD>(p, rows < ROWS_PER_LAUNCH ? rows : ROWS_PER_LAUNCH, ranks, vec, s);
        p.x += ROWS_PER_LAUNCH * p.ldx * ESZ;
        p.y += ROWS_PER_LAUNCH * p.ldy * ESZ;
        if constexpr (ADD) {
            p.r += ROWS_PER_LAUNCH * p.ldr * ESZ;
            p.s += ROWS_PER_LAUNCH * p.ldy * ESZ;
        }
    }
}

// out = a + b, rounded, for both ranks of a launch (blockIdx.y): the addition behind a decoder layer's MLP, which torch makes rank by rank (3.2-4.6 us each in a recorded
// step; one launch of 4.6-4.8 for both). Latency at the sizes that come here, so plain 16-byte chunks, one a lane. x, r: the operands; n 16-byte chunks, then the elements behind them.
template <int DT>
__global__ __launch_bounds__(256) void add_ranks_kernel(NormParams p, int64_t n, int tail) {
    take_rank(p);
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i < n) {
        const Chunk<DT> a = unpack<DT>(reinterpret_cast<const uint4 *>(p.x)[i]), b = unpack<DT>(reinterpret_cast<const uint4 *>(p.r)[i]);
        Chunk<DT> c;
#pragma unroll
        for (int e = 0; e < Chunk<DT>::E; ++e) c.v[e] = a.v[e] + b.v[e];
        reinterpret_cast<uint4 *>(p.y)[i] = pack<DT>(c);
    } else if (i - n < tail) {
        const int64_t e = n * Chunk<DT>::E + (i - n);
        if constexpr (DT == TPAMD_F32) reinterpret_cast<float *>(p.y)[e] = reinterpret_cast<const float *>(p.x)[e] + reinterpret_cast<const float *>(p.r)[e];
        else
            reinterpret_cast<uint16_t *>(p.y)[e] =
                f32_to_half<DT>(half_to_f32<DT>(reinterpret_cast<const uint16_t *>(p.x)[e]) + half_to_f32<DT>(reinterpret_cast<const uint16_t *>(p.r)[e]));
    }
}

template <int DT>
void launch_layer(NormParams p, int64_t rows, int ranks, bool vec, hipStream_t s) {
    constexpr int64_t ESZ = DT == TPAMD_F32 ? 4 : 2;
    for (; rows > 0; rows -= ROWS_PER_LAUNCH) {
        launch_layer_rows<DT>(p, rows < ROWS_PER_LAUNCH ? rows : ROWS_PER_LAUNCH, ranks, vec, s);
        p.x += ROWS_PER_LAUNCH * p.ldx * ESZ;
        p.y += ROWS_PER_LAUNCH * p.ldy * ESZ;
    }
}

}  // namespace
}  // namespace tpamd

using namespace tpamd;

// n ranks' rows of one shape, two ranks to a launch.
static int run_norm(const char *who, int n, const void *const *x, const void *const *r, const void *const *w, void *const *sum, void *const *y,
                    int64_t rows, int64_t D, int64_t ldx, int64_t ldr, int64_t ldy, float eps, int dtype, void *stream) {
    const bool add = r != nullptr;
    TPAMD_REQUIRE(n >= 0 && x && w && y && (!add || sum), "%s: null pointer", who);
    TPAMD_REQUIRE(dtype == TPAMD_BF16 || dtype == TPAMD_F16 || dtype == TPAMD_F32, "%s: unknown dtype %d", who, dtype);
    TPAMD_REQUIRE(rows >= 0 && D >= 0 && D < (1ll << 31), "%s: bad dimension", who);
    if (rows == 0 || D == 0) return TPAMD_OK;
    TPAMD_REQUIRE(ldx >= D && ldy >= D && (!add || ldr >= D), "%s: leading dimension smaller than the row", who);
    bool vec = dtype != TPAMD_F32 && D % 8 == 0 && D <= 16 * 64 * 2 * 8 && ldx % 8 == 0 && ldr % 8 == 0 && ldy % 8 == 0;
    for (int i = 0; i < n; ++i) {
        TPAMD_REQUIRE(x[i] && w[i] && y[i] && (!add || (r[i] && sum[i])), "%s: null pointer", who);
        vec = vec && aligned(x[i], 16) && aligned(w[i], 16) && aligned(y[i], 16) && (!add || (aligned(r[i], 16) && aligned(sum[i], 16)));
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    for (int i = 0; i < n; i += 2) {
        const int ranks = i + 1 < n ? 2 : 1;
        NormParams p{static_cast<const char *>(x[i]), static_cast<const char *>(w[i]), static_cast<const char *>(add ? r[i] : nullptr), static_cast<char *>(y[i]),
                     static_cast<char *>(add ? sum[i] : nullptr), ldx, ldr, ldy, static_cast<int>(D), eps, {}};
        if (ranks == 2) {
            p.to = {bytes_from(x[i], x[i + 1]), bytes_from(w[i], w[i + 1]), add ? bytes_from(r[i], r[i + 1]) : 0, bytes_from(y[i], y[i + 1]),
                    add ? bytes_from(sum[i], sum[i + 1]) : 0};
        }
        if (dtype == TPAMD_BF16) add ? launch<TPAMD_BF16, true>(p, rows, ranks, vec, s) : launch<TPAMD_BF16, false>(p, rows, ranks, vec, s);
        else if (dtype == TPAMD_F16) add ? launch<TPAMD_F16, true>(p, rows, ranks, vec, s) : launch<TPAMD_F16, false>(p, rows, ranks, vec, s);
        else add ? launch<TPAMD_F32, true>(p, rows, ranks, vec, s) : launch<TPAMD_F32, false>(p, rows, ranks, vec, s);
        TPAMD_HIP(hipGetLastError());
    }
    return TPAMD_OK;
}

extern "C" int tpamd_rms_norm(const void *x_dev, const void *w_dev, void *y_dev, int64_t rows, int64_t D, int64_t ldx, int64_t ldy,
                              float eps, int dtype, void *stream) {
    return run_norm("tpamd_rms_norm", 1, &x_dev, nullptr, &w_dev, nullptr, &y_dev, rows, D, ldx, 0, ldy, eps, dtype, stream);
}

extern "C" int tpamd_rms_norm_ranks(int n, const void *const *x_dev, const void *const *w_dev, void *const *y_dev, int64_t rows, int64_t D,
                                    int64_t ldx, int64_t ldy, float eps, int dtype, void *stream) {
    return run_norm("tpamd_rms_norm_ranks", n, x_dev, nullptr, w_dev, nullptr, y_dev, rows, D, ldx, 0, ldy, eps, dtype, stream);
}

extern "C" int tpamd_add_rms_norm(const void *x_dev, const void *r_dev, const void *w_dev, void *sum_dev, void *y_dev, int64_t rows, int64_t D,
                                  int64_t ldx, int64_t ldr, int64_t ldy, float eps, int dtype, void *stream) {
    return run_norm("tpamd_add_rms_norm", 1, &x_dev, &r_dev, &w_dev, &sum_dev, &y_dev, rows, D, ldx, ldr, ldy, eps, dtype, stream);
}

extern "C" int tpamd_add_rms_norm_ranks(int n, const void *const *x_dev, const void *const *r_dev, const void *const *w_dev, void *const *sum_dev,
                                        void *const *y_dev, int64_t rows, int64_t D, int64_t ldx, int64_t ldr, int64_t ldy, float eps, int dtype,
                                        void *stream) {
    TPAMD_REQUIRE(r_dev != nullptr, "tpamd_add_rms_norm_ranks: null pointer");
    return run_norm("tpamd_add_rms_norm_ranks", n, x_dev, r_dev, w_dev, sum_dev, y_dev, rows, D, ldx, ldr, ldy, eps, dtype, stream);
}

extern "C" int tpamd_layer_norm_ranks(int n, const void *const *x_dev, const void *const *w_dev, const void *const *b_dev, void *const *y_dev, int64_t rows,
                                      int64_t D, int64_t ldx, int64_t ldy, float eps, int dtype, void *stream) {
    const char *who = "tpamd_layer_norm_ranks";
    TPAMD_REQUIRE(n >= 0 && x_dev && w_dev && y_dev, "%s: null pointer", who);
    TPAMD_REQUIRE(dtype == TPAMD_BF16 || dtype == TPAMD_F16 || dtype == TPAMD_F32, "%s: unknown dtype %d", who, dtype);
    TPAMD_REQUIRE(rows >= 0 && D >= 0 && D < (1ll << 31), "%s: bad dimension", who);
    if (rows == 0 || D == 0) return TPAMD_OK;
    TPAMD_REQUIRE(ldx >= D && ldy >= D, "%s: leading dimension smaller than the row", who);
    const int chunk = dtype == TPAMD_F32 ? 4 : 8;
    bool vec = D % chunk == 0 && D <= 16 * 64 * 2 * chunk && ldx % chunk == 0 && ldy % chunk == 0;
    for (int i = 0; i < n; ++i) {
        TPAMD_REQUIRE(x_dev[i] && w_dev[i] && y_dev[i] && (!b_dev || b_dev[i]), "%s: null pointer", who);
        vec = vec && aligned(x_dev[i], 16) && aligned(w_dev[i], 16) && aligned(y_dev[i], 16) && (!b_dev || aligned(b_dev[i], 16));
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    for (int i = 0; i < n; i += 2) {
        const int ranks = i + 1 < n ? 2 : 1;
        NormParams p{static_cast<const char *>(x_dev[i]), static_cast<const char *>(w_dev[i]), static_cast<const char *>(b_dev ? b_dev[i] : nullptr),
                     static_cast<char *>(y_dev[i]), nullptr, ldx, 0, ldy, static_cast<int>(D), eps, {}};
        if (ranks == 2)
            p.to = {bytes_from(x_dev[i], x_dev[i + 1]), bytes_from(w_dev[i], w_dev[i + 1]), b_dev ? bytes_from(b_dev[i], b_dev[i + 1]) : 0,
                    bytes_from(y_dev[i], y_dev[i + 1]), 0};
        if (dtype == TPAMD_BF16) launch_layer<TPAMD_BF16>(p, rows, ranks, vec, s);
        else if (dtype == TPAMD_F16) launch_layer<TPAMD_F16>(p, rows, ranks, vec, s);
        else launch_layer<TPAMD_F32>(p, rows, ranks, vec, s);
        TPAMD_HIP(hipGetLastError());
    }
    return TPAMD_OK;
}

extern "C" int tpamd_add_ranks(int n, const void *const *a_dev, const void *const *b_dev, void *const *out_dev, int64_t elements, int dtype, void *stream) {
    const char *who = "tpamd_add_ranks";
    TPAMD_REQUIRE(n >= 0 && a_dev && b_dev && out_dev, "%s: null pointer", who);
    TPAMD_REQUIRE(dtype == TPAMD_BF16 || dtype == TPAMD_F16 || dtype == TPAMD_F32, "%s: unknown dtype %d", who, dtype);
    TPAMD_REQUIRE(elements >= 0 && elements < (1ll << 32), "%s: bad dimension", who);  // at most 2^31 threads in a launch of two ranks
    if (elements == 0) return TPAMD_OK;
    for (int i = 0; i < n; ++i)
        TPAMD_REQUIRE(a_dev[i] && b_dev[i] && out_dev[i] && aligned(a_dev[i], 16) && aligned(b_dev[i], 16) && aligned(out_dev[i], 16),
                      "%s: operands must be 16-byte aligned", who);
    const int per = dtype == TPAMD_F32 ? 4 : 8;
    const int64_t chunks = elements / per;
    const int tail = static_cast<int>(elements % per);
    hipStream_t s = static_cast<hipStream_t>(stream);
    for (int i = 0; i < n; i += 2) {
        const int ranks = i + 1 < n ? 2 : 1;
        NormParams p{};
        p.x = static_cast<const char *>(a_dev[i]);
        p.r = static_cast<const char *>(b_dev[i]);
        p.y = static_cast<char *>(out_dev[i]);
        if (ranks == 2) p.to = {bytes_from(a_dev[i], a_dev[i + 1]), 0, bytes_from(b_dev[i], b_dev[i + 1]), bytes_from(out_dev[i], out_dev[i + 1]), 0};
        const dim3 grid(static_cast<unsigned>((chunks + tail + 255) / 256), ranks);
        if (dtype == TPAMD_BF16) hipLaunchKernelGGL(add_ranks_kernel<TPAMD_BF16>, grid, dim3(256), 0, s, p, chunks, tail);
        else if (dtype == TPAMD_F16) hipLaunchKernelGGL(add_ranks_kernel<TPAMD_F16>, grid, dim3(256), 0, s, p, chunks, tail);
        else hipLaunchKernelGGL(add_ranks_kernel<TPAMD_F32>, grid, dim3(256), 0, s, p, chunks, tail);
        TPAMD_HIP(hipGetLastError());
    }
    return TPAMD_OK;
}
