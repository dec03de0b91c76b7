// What the weight-streaming files share: launch parameters and the stores of single outputs.
#pragma once
#include "common.h"

namespace tpamd {

enum { SK_LINEAR = 0, SK_SWIGLU = 1 };

struct SkinnyParams {
    const char *x;
    const char *w;
    const char *w2;
    const char *bias;
    const float *scale;        // int8 path: per output row
    const int *outlier_idx;    // int8 path
    const char *w_out;         // int8 path: [N, n_out] in activation dtype
    const char *addend;        // linear: added to the rounded result, or NULL
    char *y;
    int M, N, K;
    int n_out;
    int64_t ldx, ldw, ldy, ld_wout, ldadd;
    int act;
    int ranks;     // 1, or 2: blockIdx.z is the rank, `to` the way to the second one's operands
    RankStep to;
    int64_t copy;  // every output is stored a second time that many bytes on (0: once)
    int sum;       // y = round(rank 0's product) + round(rank 1's): one result for both ranks
};

// This block's rank.
__device__ __forceinline__ void take_rank(SkinnyParams &p) {
    if (blockIdx.z == 0) return;
    p.x += p.to.x; p.w += p.to.w; p.w2 += p.to.w2; p.bias += p.to.bias; p.y += p.to.y;
    p.scale = reinterpret_cast<const float *>(reinterpret_cast<const char *>(p.scale) + p.to.scale);
    p.outlier_idx = reinterpret_cast<const int *>(reinterpret_cast<const char *>(p.outlier_idx) + p.to.outlier_idx);
    p.w_out += p.to.w_out;
}

// One output element from its fp32 sums (s1 = the up sum of a gated pair): the reference's op chain with its
// roundings to the tensor dtype (gate and up products, SiLU, product), or bias and activation.
template <int DT, int MODE>
__device__ __forceinline__ void skinny_store_output(const SkinnyParams &p, float s0, float s1, int m, int n) {
    uint16_t out;
    if constexpr (MODE == SK_SWIGLU) {
        const float gv = half_to_f32<DT>(f32_to_half<DT>(s0));
        const float u = half_to_f32<DT>(f32_to_half<DT>(s1));
        const float sl = half_to_f32<DT>(f32_to_half<DT>(silu_f32(gv)));
        out = f32_to_half<DT>(sl * u);
    } else {
        float v = s0;
        if (p.bias) v += half_to_f32<DT>(reinterpret_cast<const uint16_t *>(p.bias)[n]);
        if (p.act == TPAMD_ACT_GELU) v = gelu_erf(v);
        out = f32_to_half<DT>(v);
        if (p.addend != nullptr)  // one step of the sum over rank partials: both operands in the tensor dtype
            out = f32_to_half<DT>(half_to_f32<DT>(out) + half_to_f32<DT>(reinterpret_cast<const uint16_t *>(p.addend)[static_cast<int64_t>(m) * p.ldadd + n]));
    }
    reinterpret_cast<uint16_t *>(p.y)[static_cast<int64_t>(m) * p.ldy + n] = out;
    if constexpr (MODE == SK_LINEAR) {
        if (p.copy) reinterpret_cast<uint16_t *>(p.y + p.copy)[static_cast<int64_t>(m) * p.ldy + n] = out;
    }
}

// One element of the sum of two ranks' Linears from the fp32 sums of each: products rounded to the tensor dtype, then the rounded sum, which is what
// a Linear whose epilogue adds the other's result gives.
template <int DT>
__device__ __forceinline__ void skinny_store_sum(const SkinnyParams &p, float s0, float s1, int m, int n) {
    if (p.bias) {
        s0 += half_to_f32<DT>(reinterpret_cast<const uint16_t *>(p.bias)[n]);
        s1 += half_to_f32<DT>(reinterpret_cast<const uint16_t *>(p.bias + p.to.bias)[n]);
    }
    const uint16_t out = f32_to_half<DT>(half_to_f32<DT>(f32_to_half<DT>(s0)) + half_to_f32<DT>(f32_to_half<DT>(s1)));
    reinterpret_cast<uint16_t *>(p.y)[static_cast<int64_t>(m) * p.ldy + n] = out;
    if (p.copy) reinterpret_cast<uint16_t *>(p.y + p.copy)[static_cast<int64_t>(m) * p.ldy + n] = out;
}

// stream.hip. Whether its kernel takes a Linear (swiglu: gated pair) of `ranks` matrices in one launch, or two ranks' Linears and their sum, on M rows, and
// the launch (operands of mfma_ok).
bool stream_pays(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int ranks, bool swiglu, bool sum, int cus);
int stream_dispatch(const SkinnyParams &p, int dtype, bool swiglu, hipStream_t s);
// stream_w8.hip, the same for int8 weights.
bool stream_w8_pays(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t n_out, int ranks, bool sum, int cus);
int stream_w8_dispatch(const SkinnyParams &p, int dtype, hipStream_t s);

}  // namespace tpamd
