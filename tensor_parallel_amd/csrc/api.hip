// C ABI entry points for the shard Linears, plus the library's error plumbing.
#include "common.h"
#include "gemm_model.h"

#include <string.h>

namespace tpamd {

static thread_local char g_err[512] = "";

void set_error(const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

int gemm_dispatch(const void *x, const void *w, const void *w2, const void *bias, const void *addend, int64_t ldadd, void *y,
                  int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ldy, int dtype, int act, bool swiglu,
                  bool generic, hipStream_t s, const RankStep *second = nullptr, int64_t copy = 0);
int skinny_dispatch(const void *x, const void *w, const void *w2, const void *bias, const void *addend, int64_t ldadd,
                    const void *scale, const void *outlier_idx, const void *w_out, int64_t n_out, void *y, int64_t M, int64_t N,
                    int64_t K, int64_t ldx, int64_t ldw, int64_t ldy, int64_t ld_wout, int dtype, int act, bool swiglu, bool w8,
                    hipStream_t s, const RankStep *second = nullptr, int64_t copy = 0);

bool stream_pays(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int ranks, bool swiglu, bool sum, int cus);

bool w8_direct_ok(int64_t K, int64_t ldx, int64_t ldw);
int gemm_w8_dispatch(const void *x, const void *wq, const void *scale, const void *outlier_idx, const void *w_out, int64_t n_out,
                     const void *bias, const void *addend, int64_t ldadd, int64_t copy, void *y, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw,
                     int64_t ld_wout, int64_t ldy, int dtype, int act, hipStream_t s);

int attention_dispatch(const void *q, const void *k, const void *v, void *o, int64_t B, int64_t Hq, int64_t Hkv, int64_t Sq,
                       int64_t Skv, int64_t D, const int64_t *strides, float scale, int causal, int dtype, hipStream_t s);
int attention_decode_rope_dispatch(const void *q, const void *k, const void *v, const void *cos, const void *sin, void *k_cache,
                                   void *v_cache, void *o, int64_t B, int64_t Hq, int64_t Hkv, int64_t D, int64_t pos0, const int64_t *pos_dev,
                                   const int64_t *strides, float scale, int dtype, hipStream_t s, const tpamd_decode_rank *second = nullptr);

int skinny_sum_dispatch(const void *x, const void *w, const void *bias, const RankStep &to, void *y, int64_t copy, int64_t M, int64_t N, int64_t K, int64_t ldx,
                        int64_t ldw, int64_t ldy, int dtype, int row_waves, hipStream_t s);
bool sum128_pays(int64_t M, int64_t N, int64_t K, int cus);
int gemm_sum_dispatch(const void *x, const void *w, const void *bias, const RankStep &to, void *y, int64_t copy, int64_t M, int64_t N, int64_t K, int64_t ldx,
                      int64_t ldw, int64_t ldy, int dtype, hipStream_t s, bool *done);
int skinny_w8_sum_dispatch(const void *x, const void *wq, const void *scale, const void *outlier_idx, const void *w_out, int64_t n_out, const void *bias,
                           const RankStep &to, void *y, int64_t copy, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ld_wout, int64_t ldy,
                           int dtype, hipStream_t s, bool *done);

namespace {

// Largest M served by the weight-streaming kernels; above it the tiled MFMA kernels take over.
constexpr int64_t SKINNY_MAX_M = 16;

// A single 16-bit matrix with at most one 16-column tile per CU stays with the weight-streaming kernel for more rows: the
// tiled kernels split K over blocks there and pay a second launch. How far depends on the row length. Measured inside a
// HIP graph (us, streaming / tiled) at 17 / 32 / 48 / 64 rows:
//   2048 x 2048   6.3  6.8  8.6  8.9 /  9.3  9.9 10.3 10.9     4096 x 2048   6.9  7.7 10.2 10.7 / 10.3 11.2 11.6 12.6
//   3072 x 3072   8.0  9.1 10.7 11.3 / 11.0 11.8 12.0 12.8     (K <= 3072: streaming up to 64 rows)
//   2048 x 4096   9.1 10.2 12.9 13.5 / 10.6 11.2 11.6 12.2     4096 x 4096  10.0 11.4 14.8 16.0 / 12.0 12.6 13.4 14.4
//   4096 x 5504  13.5 15.0 18.5 19.9 / 16.3 16.9 18.0 19.1     4096 x 8192  16.7 18.7 23.3 24.7 / 17.9 18.8 19.5 20.3
//                                                              (longer rows: streaming up to 32 rows)
//   2048 x 8192  14.4 16.4 21.0 22.9 / 13.2 13.9 15.1 16.0     1536 x 6144  11.8 13.6 17.1 18.5 / 11.7 12.2 12.6 13.1
//                                                              (K >= 6144 on at most half a tile per CU: tiled from 17 rows)
// Beside stream_kernel, which is asked first (decode_rows). With more tiles the tiled kernels win from 17 rows on (11008 x 4096: 26.5 29.0 36.2 39.0 / 24.6 25.4 25.3 26.5), and the
// gated pair is faster through them at all of these sizes.
int skinny_row_limit(int64_t N, int64_t K, int64_t *rows) {
    *rows = SKINNY_MAX_M;
    if (tuning().skinny_max_m != TUNE_UNSET) {
        *rows = tuning().skinny_max_m < 64 ? tuning().skinny_max_m : 64;
        return TPAMD_OK;
    }
    int dev = 0, cus = 256;
    TPAMD_HIP(hipGetDevice(&dev));
    if (int rc = device_cus(dev, &cus); rc != TPAMD_OK) return rc;
    const int64_t tiles = (N + 15) / 16;
    if (K < 2048 || K > 8192 || tiles > cus) return TPAMD_OK;
    if (K <= 3072) *rows = 64;
    else if (!(K >= 6144 && tiles * 2 <= cus)) *rows = 32;
    return TPAMD_OK;
}
// The gated pair with at most one 8-column tile per CU (2048 columns on 256 CUs) and rows of up to 6144 elements stays
// with the weight-streaming kernel up to 32 rows. Measured inside a HIP graph (us, streaming / tiled) at 17 / 24 / 32 rows:
//   1376 x 2048   6.6  6.9  7.2 / 10.7 11.5 12.3     2048 x 4096  10.8 10.9 11.6 / 12.2 12.3 12.8
//   1376 x 4096  10.3 10.3 11.0 / 12.0 12.3 13.1     2048 x 5504  13.7 14.3 15.3 / 14.6 14.9 15.4
// With more columns the tiled kernels win (2752 x 4096: 17.4 18.4 20.0 / 14.5 14.7 15.1), and on K = 8192 from 1024 columns on.
int pair_row_limit(int64_t N, int64_t K, int64_t *rows) {
    *rows = SKINNY_MAX_M;
    if (tuning().skinny_max_m != TUNE_UNSET) {
        *rows = tuning().skinny_max_m < 32 ? tuning().skinny_max_m : 32;
        return TPAMD_OK;
    }
    int dev = 0, cus = 256;
    TPAMD_HIP(hipGetDevice(&dev));
    if (int rc = device_cus(dev, &cus); rc != TPAMD_OK) return rc;
    if (K >= 2048 && K <= 6144 && (N + 7) / 8 <= cus) *rows = 32;
    return TPAMD_OK;
}
// Rows that skinny_dispatch takes of `ranks` matrices (pair: gated pairs) of N columns each in one launch: those of the kernels above, and what stream_kernel takes.
int decode_rows(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int ranks, bool pair, int64_t *rows) {
    *rows = SKINNY_MAX_M;
    if (M <= SKINNY_MAX_M || M > 64) return TPAMD_OK;
    int dev = 0, cus = 256;
    TPAMD_HIP(hipGetDevice(&dev));
    if (int rc = device_cus(dev, &cus); rc != TPAMD_OK) return rc;
    if (stream_pays(M, N, K, ldx, ldw, ranks, pair, false, cus)) {
        *rows = 64;
        return TPAMD_OK;
    }
    return pair ? (M <= 32 ? pair_row_limit(ranks * N, K, rows) : TPAMD_OK) : skinny_row_limit(ranks * N, K, rows);
}
constexpr int64_t SKINNY_W8_SLAB = 64;

// What the MFMA kernels need from 16-bit operands: 16-byte aligned rows of x and w, 8-byte aligned groups of 4
// outputs. Anything else goes to the scalar-load kernel.
bool mfma_ok(const void *x, const void *w, const void *w2, const void *bias, const void *y, int64_t N, int64_t K,
             int64_t ldx, int64_t ldw, int64_t ldy) {
    return aligned(x, 16) && aligned(w, 16) && (!w2 || aligned(w2, 16)) && aligned(y, 8) && (!bias || aligned(bias, 8)) &&
           K % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && N % 4 == 0 && ldy % 4 == 0;
}

int check_common(const char *who, const void *x, const void *w, const void *y, int64_t M, int64_t N, int64_t K,
                 int64_t ldx, int64_t ldw, int64_t ldy, int dtype) {
    TPAMD_REQUIRE(M >= 0 && N >= 0 && K >= 0, "%s: negative dimension (M=%lld N=%lld K=%lld)", who, (long long)M,
                  (long long)N, (long long)K);
    TPAMD_REQUIRE(M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31), "%s: dimension over 2^31", who);
    TPAMD_REQUIRE(dtype == TPAMD_BF16 || dtype == TPAMD_F16 || dtype == TPAMD_F32, "%s: unknown dtype %d", who, dtype);
    if (M == 0 || N == 0) return TPAMD_OK;
    TPAMD_REQUIRE(x && w && y, "%s: null pointer", who);
    TPAMD_REQUIRE(ldx >= K && ldw >= K && ldy >= N, "%s: leading dimension smaller than the row (ldx=%lld ldw=%lld ldy=%lld)",
                  who, (long long)ldx, (long long)ldw, (long long)ldy);
    return TPAMD_OK;
}

}  // namespace
}  // namespace tpamd

using namespace tpamd;

extern "C" int tpamd_abi_version(void) { return TPAMD_ABI_VERSION; }
extern "C" const char *tpamd_last_error(void) { return g_err; }

// y = act(x . w^T + bias), then, with an addend, y = round(y + addend) in the tensor dtype.
int tpamd::linear_entry(const char *who, const void *x_dev, const void *w_dev, const void *bias_dev, const void *addend_dev,
                        int64_t ldadd, void *y_dev, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ldy,
                        int dtype, int act, void *stream, void *copy_dev) {
    int rc = check_common(who, x_dev, w_dev, y_dev, M, N, K, ldx, ldw, ldy, dtype);
    if (rc != TPAMD_OK) return rc;
    TPAMD_REQUIRE(act == TPAMD_ACT_NONE || act == TPAMD_ACT_GELU, "%s: unknown activation %d", who, act);
    if (M == 0 || N == 0) return TPAMD_OK;
    TPAMD_REQUIRE(addend_dev == nullptr || ldadd >= N, "%s: ldadd=%lld is smaller than N=%lld", who, (long long)ldadd, (long long)N);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool fast = dtype != TPAMD_F32 && mfma_ok(x_dev, w_dev, nullptr, bias_dev, y_dev, N, K, ldx, ldw, ldy) &&
                      (addend_dev == nullptr || (aligned(addend_dev, 8) && ldadd % 4 == 0)) && aligned(copy_dev, 8);
    const int64_t copy = bytes_from(y_dev, copy_dev);
    int64_t skinny_rows = SKINNY_MAX_M;
    if (fast) {
        rc = decode_rows(M, N, K, ldx, ldw, 1, false, &skinny_rows);
        if (rc != TPAMD_OK) return rc;
    }
    if (fast && M <= skinny_rows)
        return skinny_dispatch(x_dev, w_dev, nullptr, bias_dev, addend_dev, ldadd, nullptr, nullptr, nullptr, 0, y_dev, M, N, K,
                               ldx, ldw, ldy, 0, dtype, act, false, false, s, nullptr, copy);
    return gemm_dispatch(x_dev, w_dev, nullptr, bias_dev, addend_dev, ldadd, y_dev, M, N, K, ldx, ldw, ldy, dtype, act, false,
                         !fast, s, nullptr, copy);
}

extern "C" int tpamd_linear(const void *x_dev, const void *w_dev, const void *bias_dev, void *y_dev, int64_t M, int64_t N,
                            int64_t K, int64_t ldx, int64_t ldw, int64_t ldy, int dtype, int act, void *stream) {
    return linear_entry("tpamd_linear", x_dev, w_dev, bias_dev, nullptr, 0, y_dev, M, N, K, ldx, ldw, ldy, dtype, act, stream);
}

extern "C" int tpamd_linear_add(const void *x_dev, const void *w_dev, const void *bias_dev, const void *addend_dev, void *y_dev,
                                int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ldadd, int64_t ldy, int dtype,
                                int act, void *stream) {
    TPAMD_REQUIRE(addend_dev != nullptr || M == 0 || N == 0, "tpamd_linear_add: addend is NULL");
    return linear_entry("tpamd_linear_add", x_dev, w_dev, bias_dev, addend_dev, ldadd, y_dev, M, N, K, ldx, ldw, ldy, dtype, act,
                        stream);
}

// The second store instead of a copying launch behind the sum (2.9 us for one row of 4096, 4.7 for 8, 6.2 for 2103, four in a recorded step of two
// layers): 8 rows on 2048 positions 423 -> 409 us, with the head's gather.
extern "C" int tpamd_linear_add_copy(const void *x_dev, const void *w_dev, const void *bias_dev, const void *addend_dev, void *y_dev, void *copy_dev,
                                     int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ldadd, int64_t ldy, int dtype, int act,
                                     void *stream) {
    TPAMD_REQUIRE((addend_dev != nullptr && copy_dev != nullptr && copy_dev != y_dev) || M == 0 || N == 0,
                  "tpamd_linear_add_copy: the addend or the copy is NULL, or the copy is y");
    return linear_entry("tpamd_linear_add_copy", x_dev, w_dev, bias_dev, addend_dev, ldadd, y_dev, M, N, K, ldx, ldw, ldy, dtype, act,
                        stream, copy_dev);
}

extern "C" int tpamd_swiglu_up(const void *x_dev, const void *wg_dev, const void *wu_dev, void *h_dev, int64_t M, int64_t N,
                               int64_t K, int64_t ldx, int64_t ldw, int64_t ldh, int dtype, void *stream) {
    int rc = check_common("tpamd_swiglu_up", x_dev, wg_dev, h_dev, M, N, K, ldx, ldw, ldh, dtype);
    if (rc != TPAMD_OK) return rc;
    if (M == 0 || N == 0) return TPAMD_OK;
    TPAMD_REQUIRE(wu_dev != nullptr, "tpamd_swiglu_up: wu is NULL");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool fast = dtype != TPAMD_F32 && mfma_ok(x_dev, wg_dev, wu_dev, nullptr, h_dev, N, K, ldx, ldw, ldh);
    int64_t pair_rows = SKINNY_MAX_M;
    if (fast) {
        rc = decode_rows(M, N, K, ldx, ldw, 1, true, &pair_rows);
        if (rc != TPAMD_OK) return rc;
    }
    if (fast && M <= pair_rows)
        return skinny_dispatch(x_dev, wg_dev, wu_dev, nullptr, nullptr, 0, nullptr, nullptr, nullptr, 0, h_dev, M, N, K, ldx, ldw,
                               ldh, 0, dtype, TPAMD_ACT_NONE, true, false, s);
    return gemm_dispatch(x_dev, wg_dev, wu_dev, nullptr, nullptr, 0, h_dev, M, N, K, ldx, ldw, ldh, dtype, TPAMD_ACT_NONE, true,
                         !fast, s);
}

// n ranks' Linears (w2: gated pairs) of one shape, two to a launch where both have what the fast kernels need. A rank's half of a decode-sized
// matrix streams at 3-5.7 TB/s because a launch starts and drains in about 2 us; both halves in one reach 5.5-6.7. Two launches / one, in a
// recorded decode step (us, kernel trace, bf16, one row): QKV 6144 x 4096 21.0 / 16.4, the pair 5504 x 4096 31.6 / 28.4, head 16000 x 4096
// 41.2 / 39.1; 40 rows in fp16: the pair 58.4 (two K splits and their finishing launches) / 40.2 (unsplit, its tiles now fill the device),
// QKV 3072 x 4096 27.8 / 17.9 a rank; 512 rows: the pair 106 / 104 (464 tiles of 128 x 192: 1.8 rounds for twice 0.9).
static int matmul_ranks(const char *who, int n, const void *const *x, const void *const *w, const void *const *w2, const void *const *bias,
                        void *const *y, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ldy, int dtype, int act, void *stream) {
    TPAMD_REQUIRE(n >= 0 && x && w && y, "%s: null pointer", who);
    const bool pair = w2 != nullptr;
    auto single = [&](int i) {
        return pair ? tpamd_swiglu_up(x[i], w[i], w2[i], y[i], M, N, K, ldx, ldw, ldy, dtype, stream)
                    : linear_entry(who, x[i], w[i], bias ? bias[i] : nullptr, nullptr, 0, y[i], M, N, K, ldx, ldw, ldy, dtype, act, stream);
    };
    for (int i = 0; i < n; ++i) {
        const void *b0 = bias ? bias[i] : nullptr, *b1 = bias && i + 1 < n ? bias[i + 1] : nullptr;
        bool both = i + 1 < n && M > 0 && N > 0 && dtype != TPAMD_F32 && (b0 == nullptr) == (b1 == nullptr) && (act == TPAMD_ACT_NONE || act == TPAMD_ACT_GELU);
        for (int j = i; both && j < i + 2; ++j) {
            if (int rc = check_common(who, x[j], w[j], y[j], M, N, K, ldx, ldw, ldy, dtype); rc != TPAMD_OK) return rc;
            TPAMD_REQUIRE(!pair || w2[j] != nullptr, "%s: null pointer", who);
            both = mfma_ok(x[j], w[j], pair ? w2[j] : nullptr, j == i ? b0 : b1, y[j], N, K, ldx, ldw, ldy);
        }
        if (!both) {
            if (int rc = single(i); rc != TPAMD_OK) return rc;
            continue;
        }
        RankStep to{};
        to.x = bytes_from(x[i], x[i + 1]);
        to.w = bytes_from(w[i], w[i + 1]);
        to.w2 = pair ? bytes_from(w2[i], w2[i + 1]) : 0;
        to.bias = bytes_from(b0, b1);
        to.y = bytes_from(y[i], y[i + 1]);
        int64_t rows = SKINNY_MAX_M;
        if (int rc = decode_rows(M, N, K, ldx, ldw, 2, pair, &rows); rc != TPAMD_OK) return rc;
        const int rc = M <= rows ? skinny_dispatch(x[i], w[i], pair ? w2[i] : nullptr, b0, nullptr, 0, nullptr, nullptr, nullptr, 0, y[i], M, N, K, ldx, ldw,
                                                   ldy, 0, dtype, act, pair, false, static_cast<hipStream_t>(stream), &to)
                                 : gemm_dispatch(x[i], w[i], pair ? w2[i] : nullptr, b0, nullptr, 0, y[i], M, N, K, ldx, ldw, ldy, dtype, act, pair, false,
                                                 static_cast<hipStream_t>(stream), &to);
        if (rc != TPAMD_OK) return rc;
        ++i;
    }
    return TPAMD_OK;
}

extern "C" int tpamd_linear_ranks(int n, const void *const *x_dev, const void *const *w_dev, const void *const *bias_dev, void *const *y_dev, int64_t M,
                                  int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ldy, int dtype, int act, void *stream) {
    return matmul_ranks("tpamd_linear_ranks", n, x_dev, w_dev, nullptr, bias_dev, y_dev, M, N, K, ldx, ldw, ldy, dtype, act, stream);
}

extern "C" int tpamd_swiglu_up_ranks(int n, const void *const *x_dev, const void *const *wg_dev, const void *const *wu_dev, void *const *h_dev, int64_t M,
                                     int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ldh, int dtype, void *stream) {
    TPAMD_REQUIRE(wu_dev != nullptr, "tpamd_swiglu_up_ranks: wu is NULL");
    return matmul_ranks("tpamd_swiglu_up_ranks", n, x_dev, wg_dev, wu_dev, nullptr, h_dev, M, N, K, ldx, ldw, ldh, dtype, TPAMD_ACT_NONE, stream);
}

// Column-parallel Linears of n ranks, each rank's columns written into every rank's whole output: two launches and a concatenation in one. What bounded
// the small ones was launches: fp32 [128 x 768] by two halves of 384 columns 13.0 + 13.0 + 7.7 us, now 13.9; OPT-125m on 2 x 64 tokens, 72 of them,
// 445 -> 300 launches and 7.66 -> 5.37 ms eager (kernels 3.4 -> 2.0 ms). A recorded decode step's output head on one row 20.6 + 20.6 + 4.8 -> 37.9 us.
extern "C" int tpamd_linear_gather_ranks(int n, const void *const *x_dev, const void *const *w_dev, const void *const *bias_dev, void *const *y_dev,
                                         int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ldy, int dtype, int act, void *stream) {
    const char *who = "tpamd_linear_gather_ranks";
    TPAMD_REQUIRE(n >= 0 && (n == 0 || (x_dev && w_dev && y_dev)), "%s: null pointer", who);
    TPAMD_REQUIRE(dtype == TPAMD_BF16 || dtype == TPAMD_F16 || dtype == TPAMD_F32, "%s: unknown dtype %d", who, dtype);
    TPAMD_REQUIRE(act == TPAMD_ACT_NONE || act == TPAMD_ACT_GELU, "%s: unknown activation %d", who, act);
    const int64_t esz = dtype == TPAMD_F32 ? 4 : 2;
    bool fast = n == 2 && M > 0 && N > 0 && (bias_dev == nullptr || (bias_dev[0] == nullptr) == (bias_dev[1] == nullptr));
    for (int i = 0; i < n; ++i) {
        const void *b = bias_dev ? bias_dev[i] : nullptr;
        if (int rc = check_common(who, x_dev[i], w_dev[i], y_dev[i], M, N, K, ldx, ldw, ldy, dtype); rc != TPAMD_OK) return rc;
        TPAMD_REQUIRE(M == 0 || N == 0 || ldy >= n * N, "%s: ldy=%lld does not hold %d ranks' columns", who, (long long)ldy, n);
        fast = fast && (dtype == TPAMD_F32 ? aligned(x_dev[i], 16) && aligned(w_dev[i], 16) && aligned(y_dev[i], 16) && aligned(b, 16) && K >= 4 && K % 4 == 0 &&
                                                 N % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && ldy % 4 == 0
                                           : mfma_ok(x_dev[i], w_dev[i], nullptr, b, y_dev[i], N, K, ldx, ldw, ldy));
    }
    if (M == 0 || N == 0) return TPAMD_OK;
    if (!fast) {  // rank by rank into the first output, which is then copied
        for (int i = 0; i < n; ++i) {
            const int rc = linear_entry(who, x_dev[i], w_dev[i], bias_dev ? bias_dev[i] : nullptr, nullptr, 0, static_cast<char *>(y_dev[0]) + i * N * esz, M, N, K,
                                        ldx, ldw, ldy, dtype, act, stream);
            if (rc != TPAMD_OK) return rc;
        }
        for (int i = 1; i < n; ++i) {
            const uint64_t pitch = static_cast<uint64_t>(ldy * esz);
            const tpamd_copy_job job = {y_dev[0], y_dev[i], static_cast<uint64_t>(M), static_cast<uint64_t>(n * N * esz), pitch, pitch};
            if (int rc = tpamd_copy_jobs_run(&job, 1, stream); rc != TPAMD_OK) return rc;
        }
        return TPAMD_OK;
    }
    const void *b0 = bias_dev ? bias_dev[0] : nullptr, *b1 = bias_dev ? bias_dev[1] : nullptr;
    RankStep to{};
    to.x = bytes_from(x_dev[0], x_dev[1]);
    to.w = bytes_from(w_dev[0], w_dev[1]);
    to.bias = bytes_from(b0, b1);
    to.y = N * esz;
    const int64_t copy = bytes_from(y_dev[0], y_dev[1]);
    hipStream_t s = static_cast<hipStream_t>(stream);
    int64_t rows = dtype == TPAMD_F32 ? 0 : SKINNY_MAX_M;
    if (dtype != TPAMD_F32) {
        if (int rc = decode_rows(M, N, K, ldx, ldw, 2, false, &rows); rc != TPAMD_OK) return rc;
    }
    if (M <= rows)
        return skinny_dispatch(x_dev[0], w_dev[0], nullptr, b0, nullptr, 0, nullptr, nullptr, nullptr, 0, y_dev[0], M, N, K, ldx, ldw, ldy, 0, dtype, act, false,
                               false, s, &to, copy);
    return gemm_dispatch(x_dev[0], w_dev[0], nullptr, b0, nullptr, 0, y_dev[0], M, N, K, ldx, ldw, ldy, dtype, act, false, false, s, &to, copy);
}

// What takes the sum of two ranks' row-parallel Linears: stream_kernel at 2 to 64 rows where it is the faster one (stream_model.h: 3 to 16 rows of whole 64-element units always, 4096 x 5504 at 16 rows
// 20.3 us, 22.1 by what follows), else what follows. Measured inside a HIP graph on rotated weights against tpamd_linear + tpamd_linear_add_copy (us, two
// launches / row kernel with 8 wavefronts / with 16 / MFMA weight streaming / K ranges of 128 x 128 tiles):
//   1 row    4096 x 2048   9.4 /  7.1  7.2            4096 x 5504 19.2 / 18.6 17.6     8192 x 4096 24.1 / 23.5 22.7     1024 x 1408 5.8 / 3.4  4.4
//   2 rows   4096 x 2048  10.2 /  8.3  8.7            4096 x 5504 20.3 / 22.2 43.1     8192 x 4096 26.5 / 30.4 41.9     2048 x 2816 10.0 / 7.6 11.5
//   4 rows   4096 x 2048  12.0 /           9.3        4096 x 5504 23.0 /      19.7     8192 x 4096 28.4 /      23.8     2048 x 2816 11.7 /      8.3
//   16 rows  4096 x 2048  13.4 /          10.1        4096 x 5504 25.2 /      21.5     8192 x 4096 30.6 /      27.1     5120 x 6912 34.5 / 39.3, 31.1 in tiles
//   40 rows  4096 x 2048  19.9 /               14.0   4096 x 5504 35.3 /      26.8     8192 x 4096 38.3 /      35.4     5120 x 6912 40.8 /      32.2
// So beside stream_kernel the row kernel takes one row, and two where they are short or few; weight streaming the others up to the row count it has for one matrix of both ranks' K,
// unless its tiles are a ragged number of rounds; K ranges of tiles the rest, above 64 rows while they are predicted to be faster than two launches. What stays in two
// launches and why: sum_in_two_launches (gemm_model.h).
enum SumPath { SUM_NONE, SUM_STREAM, SUM_ROWS8, SUM_ROWS16, SUM_SKINNY, SUM_TILES };
static int sum_path(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, SumPath *path) {
    *path = SUM_NONE;
    int dev = 0, cus = 256;
    TPAMD_HIP(hipGetDevice(&dev));
    if (int rc = device_cus(dev, &cus); rc != TPAMD_OK) return rc;
    if (stream_pays(M, N, K, ldx, ldw, 2, false, true, cus)) {
        *path = SUM_STREAM;
        return TPAMD_OK;
    }
    if (sum_in_two_launches(M, N, K, cus)) return TPAMD_OK;
    const int64_t tiles = (N + 15) / 16;
    const bool ragged = tiles > cus && tiles % cus != 0;
    if (K <= 11 * 512 && (M == 1 || (M == 2 && (K <= 2048 || N <= 2048)) || (M == 3 && K <= 2048 && N <= 1024))) {
        *path = M == 1 && K > 2048 && N >= 4096 ? SUM_ROWS16 : SUM_ROWS8;
        return TPAMD_OK;
    }
    int64_t rows = SKINNY_MAX_M;
    if (M > SKINNY_MAX_M && M <= 64) {
        if (int rc = skinny_row_limit(N, 2 * K, &rows); rc != TPAMD_OK) return rc;
    }
    if (M <= rows && !ragged) *path = SUM_SKINNY;
    else if (M <= 64 ? K % 64 == 0 && (N + 127) / 128 * 2 <= 4ll * cus : sum128_pays(M, N, K, cus)) *path = SUM_TILES;  // (the tiles that scratch memory holds)
    return TPAMD_OK;
}

extern "C" int tpamd_linear_sum_pays(int64_t M, int64_t N, int64_t K, int dtype) {
    SumPath path = SUM_NONE;
    return dtype != TPAMD_F32 && sum_path(M, N, K, K, K, &path) == TPAMD_OK && path != SUM_NONE ? 1 : 0;
}

// Row-parallel Linears of two ranks and their sum, delivered to both. TPAMD_ERR_UNSUPPORTED, with nothing launched, where two launches
// (tpamd_linear, then tpamd_linear_add_copy) are the better way or the kernels do not take the operands.
extern "C" int tpamd_linear_sum_ranks(const void *const *x_dev, const void *const *w_dev, const void *const *bias_dev, void *const *y_dev, int64_t M, int64_t N,
                                      int64_t K, int64_t ldx, int64_t ldw, int64_t ldy, int dtype, void *stream) {
    const char *who = "tpamd_linear_sum_ranks";
    TPAMD_REQUIRE(x_dev && w_dev && y_dev, "%s: null pointer", who);
    bool fast = dtype != TPAMD_F32 && M > 0 && N > 0 && (bias_dev == nullptr || (bias_dev[0] == nullptr) == (bias_dev[1] == nullptr));
    for (int i = 0; i < 2; ++i) {
        if (int rc = check_common(who, x_dev[i], w_dev[i], y_dev[i], M, N, K, ldx, ldw, ldy, dtype); rc != TPAMD_OK) return rc;
        fast = fast && mfma_ok(x_dev[i], w_dev[i], nullptr, bias_dev ? bias_dev[i] : nullptr, y_dev[i], N, K, ldx, ldw, ldy);
    }
    if (M == 0 || N == 0) return TPAMD_OK;
    SumPath path = SUM_NONE;
    if (fast) {
        if (int rc = sum_path(M, N, K, ldx, ldw, &path); rc != TPAMD_OK) return rc;
    }
    if (path != SUM_NONE) {
        const void *b0 = bias_dev ? bias_dev[0] : nullptr, *b1 = bias_dev ? bias_dev[1] : nullptr;
        RankStep to{};
        to.x = bytes_from(x_dev[0], x_dev[1]);
        to.w = bytes_from(w_dev[0], w_dev[1]);
        to.bias = bytes_from(b0, b1);
        const int64_t copy = bytes_from(y_dev[0], y_dev[1]);
        hipStream_t s = static_cast<hipStream_t>(stream);
        if (path != SUM_TILES)
            return skinny_sum_dispatch(x_dev[0], w_dev[0], b0, to, y_dev[0], copy, M, N, K, ldx, ldw, ldy, dtype,
                                       path == SUM_ROWS8 ? 8 : path == SUM_ROWS16 ? 16 : 0, s);
        bool done = false;
        const int rc = gemm_sum_dispatch(x_dev[0], w_dev[0], b0, to, y_dev[0], copy, M, N, K, ldx, ldw, ldy, dtype, s, &done);
        if (rc != TPAMD_OK || done) return rc;
    }
    set_error("%s: no launch of both ranks for this shape", who);
    return TPAMD_ERR_UNSUPPORTED;
}

// The same for int8 weights on 2 to 64 rows: stream_w8_kernel, or kernels that split K over blocks.
extern "C" int tpamd_linear_w8_sum_ranks(const tpamd_w8_rank *ranks, int64_t n_out, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ld_wout,
                                         int64_t ldy, int dtype, void *stream) {
    const char *who = "tpamd_linear_w8_sum_ranks";
    TPAMD_REQUIRE(ranks != nullptr, "%s: null pointer", who);
    bool ok = M > 0 && M <= SKINNY_W8_SLAB && N > 0 && n_out >= 0 && n_out <= K && K < (1ll << 31) && N < (1ll << 31) && (dtype == TPAMD_BF16 || dtype == TPAMD_F16) &&
              K % 16 == 0 && ldw % 16 == 0 && ldx % 8 == 0 && ldx >= K && ldw >= K && ldy >= N && (n_out == 0 || ld_wout >= n_out) && tuning().w8_tile == TUNE_UNSET;
    for (int j = 0; ok && j < 2; ++j) {
        const tpamd_w8_rank &r = ranks[j];
        ok = r.x && r.wq && r.scale && r.y && aligned(r.x, 16) && aligned(r.wq, 16) && (n_out == 0 || (r.outlier_idx && r.w_out)) &&
             (r.bias == nullptr) == (ranks[0].bias == nullptr);
    }
    if (ok) {
        const tpamd_w8_rank &a = ranks[0], &b = ranks[1];
        const bool o = n_out > 0;
        const RankStep to = {bytes_from(a.x, b.x), bytes_from(a.wq, b.wq), 0, bytes_from(a.bias, b.bias), 0,
                             bytes_from(a.scale, b.scale), o ? bytes_from(a.outlier_idx, b.outlier_idx) : 0, o ? bytes_from(a.w_out, b.w_out) : 0};
        bool done = false;
        const int rc = skinny_w8_sum_dispatch(a.x, a.wq, a.scale, a.outlier_idx, a.w_out, n_out, a.bias, to, a.y, bytes_from(a.y, b.y), M, N, K, ldx, ldw, ld_wout,
                                              ldy, dtype, static_cast<hipStream_t>(stream), &done);
        if (rc != TPAMD_OK || done) return rc;
    }
    set_error("%s: no launch of both ranks for this shape", who);
    return TPAMD_ERR_UNSUPPORTED;
}

extern "C" int tpamd_attention(const void *q_dev, const void *k_dev, const void *v_dev, void *out_dev, int64_t B, int64_t Hq,
                               int64_t Hkv, int64_t Sq, int64_t Skv, int64_t D, const int64_t *strides, float scale, int causal,
                               int dtype, void *stream) {
    const char *who = "tpamd_attention";
    TPAMD_REQUIRE(dtype == TPAMD_BF16 || dtype == TPAMD_F16, "%s: dtype must be BF16 or F16", who);
    TPAMD_REQUIRE(B >= 0 && Hq > 0 && Hkv > 0 && Sq >= 0 && Skv >= 0, "%s: bad dimension", who);
    TPAMD_REQUIRE(Hq % Hkv == 0, "%s: %lld query heads are not a multiple of %lld key/value heads", who, (long long)Hq, (long long)Hkv);
    TPAMD_REQUIRE(strides != nullptr, "%s: strides is NULL", who);
    TPAMD_REQUIRE(!causal || Skv >= Sq, "%s: causal attention needs Skv >= Sq", who);
    if (B == 0 || Sq == 0) return TPAMD_OK;
    TPAMD_REQUIRE(Skv > 0, "%s: no keys", who);
    TPAMD_REQUIRE(q_dev && k_dev && v_dev && out_dev, "%s: null pointer", who);
    TPAMD_REQUIRE(Hq * Sq / Hkv < (1ll << 30) && Skv < (1ll << 30), "%s: sequence too long", who);
    bool ok = (D == 64 || D == 128) && aligned(q_dev, 16) && aligned(k_dev, 16) && aligned(v_dev, 16) && aligned(out_dev, 8);
    for (int i = 0; i < 9; ++i) ok = ok && strides[i] % 8 == 0;   // 16-byte loads of q, k, v rows
    for (int i = 9; i < 12; ++i) ok = ok && strides[i] % 4 == 0;  // 8-byte stores
    if (!ok) {
        set_error("%s: head_dim must be 64 or 128 and rows 16-byte aligned", who);
        return TPAMD_ERR_UNSUPPORTED;
    }
    return attention_dispatch(q_dev, k_dev, v_dev, out_dev, B, Hq, Hkv, Sq, Skv, D, strides, scale, causal, dtype,
                              static_cast<hipStream_t>(stream));
}

// What a decode step needs of its arguments; *empty: nothing to do.
static int check_decode(const char *who, const tpamd_decode_rank &r, int64_t B, int64_t Hq, int64_t Hkv, int64_t D, int64_t pos0, int64_t cache_len,
                        const int64_t *strides, int dtype, bool devpos, bool *empty) {
    *empty = false;
    TPAMD_REQUIRE(dtype == TPAMD_BF16 || dtype == TPAMD_F16, "%s: dtype must be BF16 or F16", who);
    TPAMD_REQUIRE(B >= 0 && Hq > 0 && Hkv > 0, "%s: bad dimension", who);
    TPAMD_REQUIRE(Hq % Hkv == 0, "%s: %lld query heads are not a multiple of %lld key/value heads", who, (long long)Hq, (long long)Hkv);
    if (devpos) {
        TPAMD_REQUIRE(cache_len > 0 && cache_len < (1ll << 30), "%s: the caches must hold between 1 and 2^30 positions", who);
    } else {
        TPAMD_REQUIRE(pos0 >= 0 && pos0 < cache_len, "%s: position %lld does not fit a cache of %lld positions", who, (long long)pos0,
                      (long long)cache_len);
    }
    TPAMD_REQUIRE(strides != nullptr, "%s: strides is NULL", who);
    if (B == 0) {
        *empty = true;
        return TPAMD_OK;
    }
    TPAMD_REQUIRE(r.q && r.k && r.v && r.cos && r.sin && r.k_cache && r.v_cache && r.out && (!devpos || r.pos), "%s: null pointer", who);
    TPAMD_REQUIRE(Hq / Hkv < (1ll << 20), "%s: too many query heads per key/value head", who);
    TPAMD_REQUIRE(devpos || pos0 < (1ll << 30), "%s: sequence too long", who);
    bool ok = (D == 64 || D == 128) && aligned(r.q, 16) && aligned(r.k, 16) && aligned(r.v, 16) && aligned(r.cos, 16) && aligned(r.sin, 16) &&
              aligned(r.k_cache, 16) && aligned(r.v_cache, 16) && aligned(r.out, 8) && aligned(r.pos, 8);
    for (int i = 0; i < 14; ++i) ok = ok && strides[i] % 8 == 0;   // 16-byte loads of every row
    for (int i = 14; i < 16; ++i) ok = ok && strides[i] % 4 == 0;  // 8-byte stores
    if (!ok) {
        set_error("%s: head_dim must be 64 or 128 and rows 16-byte aligned", who);
        return TPAMD_ERR_UNSUPPORTED;
    }
    return TPAMD_OK;
}

extern "C" int tpamd_attention_decode_rope(const void *q_dev, const void *k_dev, const void *v_dev, const void *cos_dev,
                                           const void *sin_dev, void *k_cache_dev, void *v_cache_dev, void *out_dev, int64_t B,
                                           int64_t Hq, int64_t Hkv, int64_t D, int64_t pos0, int64_t cache_len,
                                           const int64_t *strides, float scale, int dtype, void *stream) {
    const tpamd_decode_rank r = {q_dev, k_dev, v_dev, cos_dev, sin_dev, k_cache_dev, v_cache_dev, out_dev, nullptr};
    bool empty = false;
    const int rc = check_decode("tpamd_attention_decode_rope", r, B, Hq, Hkv, D, pos0, cache_len, strides, dtype, false, &empty);
    if (rc != TPAMD_OK || empty) return rc;
    return attention_decode_rope_dispatch(q_dev, k_dev, v_dev, cos_dev, sin_dev, k_cache_dev, v_cache_dev, out_dev, B, Hq, Hkv, D,
                                          pos0, nullptr, strides, scale, dtype, static_cast<hipStream_t>(stream));
}

extern "C" int tpamd_attention_decode_rope_devpos(const void *q_dev, const void *k_dev, const void *v_dev, const void *cos_dev,
                                                  const void *sin_dev, void *k_cache_dev, void *v_cache_dev, void *out_dev,
                                                  int64_t B, int64_t Hq, int64_t Hkv, int64_t D, const int64_t *pos_dev,
                                                  int64_t cache_len, const int64_t *strides, float scale, int dtype,
                                                  void *stream) {
    const tpamd_decode_rank r = {q_dev, k_dev, v_dev, cos_dev, sin_dev, k_cache_dev, v_cache_dev, out_dev, pos_dev};
    bool empty = false;
    const int rc = check_decode("tpamd_attention_decode_rope_devpos", r, B, Hq, Hkv, D, 0, cache_len, strides, dtype, true, &empty);
    if (rc != TPAMD_OK || empty) return rc;
    return attention_decode_rope_dispatch(q_dev, k_dev, v_dev, cos_dev, sin_dev, k_cache_dev, v_cache_dev, out_dev, B, Hq, Hkv, D,
                                          cache_len, pos_dev, strides, scale, dtype, static_cast<hipStream_t>(stream));
}

extern "C" int tpamd_attention_decode_rope_ranks(int n, const tpamd_decode_rank *ranks, int64_t B, int64_t Hq, int64_t Hkv, int64_t D, int64_t pos0,
                                                 int64_t cache_len, const int64_t *strides, float scale, int dtype, void *stream) {
    const char *who = "tpamd_attention_decode_rope_ranks";
    TPAMD_REQUIRE(n >= 0 && (n == 0 || ranks != nullptr), "%s: null pointer", who);
    for (int i = 0; i < n; ++i) {
        TPAMD_REQUIRE((ranks[i].pos != nullptr) == (ranks[0].pos != nullptr), "%s: the count is on the device for every rank or for none", who);
        bool empty = false;
        const int rc = check_decode(who, ranks[i], B, Hq, Hkv, D, pos0, cache_len, strides, dtype, ranks[0].pos != nullptr, &empty);
        if (rc != TPAMD_OK || empty) return rc;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto step = [&](const tpamd_decode_rank &r, const tpamd_decode_rank *second) {
        return attention_decode_rope_dispatch(r.q, r.k, r.v, r.cos, r.sin, r.k_cache, r.v_cache, r.out, B, Hq, Hkv, D, r.pos ? cache_len : pos0, r.pos,
                                              strides, scale, dtype, s, second);
    };
    for (int i = 0; i < n; ++i) {
        if (i + 1 < n && B * Hkv * 2 < 65536) {
            const int rc = step(ranks[i], &ranks[i + 1]);
            if (rc == TPAMD_OK) ++i;
            if (rc == TPAMD_OK) continue;
            if (rc != TPAMD_ERR_UNSUPPORTED) return rc;  // else nothing was launched: no scratch memory, or too little for two
        }
        if (int rc = step(ranks[i], nullptr); rc != TPAMD_OK) return rc;
    }
    return TPAMD_OK;
}

// The int8 Linear, with an addend (another rank's partial sum) added to the rounded result, and that stored to `copy_dev` too (NULL: not).
static int w8_entry(const char *who, const void *x_dev, const void *wq_dev, const void *scale_dev, const void *outlier_idx_dev, const void *w_out_dev,
                    int64_t n_out, const void *bias_dev, const void *addend_dev, int64_t ldadd, void *y_dev, void *copy_dev, int64_t M, int64_t N, int64_t K,
                    int64_t ldx, int64_t ldw, int64_t ld_wout, int64_t ldy, int dtype, int act, void *stream) {
    TPAMD_REQUIRE(dtype == TPAMD_BF16 || dtype == TPAMD_F16, "%s: dtype must be BF16 or F16", who);
    TPAMD_REQUIRE(M >= 0 && N >= 0 && K >= 0 && n_out >= 0, "%s: negative dimension", who);
    TPAMD_REQUIRE(M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31), "%s: dimension over 2^31", who);
    TPAMD_REQUIRE(act == TPAMD_ACT_NONE || act == TPAMD_ACT_GELU, "%s: unknown activation %d", who, act);
    if (M == 0 || N == 0) return TPAMD_OK;
    TPAMD_REQUIRE(x_dev && wq_dev && scale_dev && y_dev, "%s: null pointer", who);
    TPAMD_REQUIRE(n_out == 0 || (outlier_idx_dev && w_out_dev && ld_wout >= n_out), "%s: outlier arguments inconsistent", who);
    TPAMD_REQUIRE(n_out <= K, "%s: more outlier columns (%lld) than K", who, (long long)n_out);
    TPAMD_REQUIRE(aligned(x_dev, 16) && aligned(wq_dev, 16), "%s: x and wq must be 16-byte aligned", who);
    TPAMD_REQUIRE(K % 16 == 0 && ldw % 16 == 0 && ldx % 8 == 0, "%s: K, ldw multiples of 16 and ldx of 8 required", who);
    TPAMD_REQUIRE(ldx >= K && ldw >= K && ldy >= N, "%s: leading dimension smaller than the row", who);
    TPAMD_REQUIRE(addend_dev == nullptr || ldadd >= N, "%s: ldadd=%lld is smaller than N=%lld", who, (long long)ldadd, (long long)N);
    const int64_t copy = bytes_from(y_dev, copy_dev);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int esz = 2;
    // The weight-streaming kernels take slabs of 64 rows; above one slab the weights go through the matrix pipe once, converted
    // on their way, with packed stores that want groups of 4 outputs on 8-byte boundaries. Measured inside a HIP graph (us,
    // slabs / tiled) at 65, 100 and 129 rows:
    //   16384 x 8192  78  119  133 / 50  57  77     8192 x 16384  80  93 131 / 54  57  76     8192 x 4096  35  55  62 / 28  31  36
    //    4096 x 5504  27   36   45 / 28  29  33      4096 x 4096  22  31  39 / 26  29  30     2048 x 2048  14  19  23 / 20  22  23
    // so small matrices stay with the slabs while the second one is nearly empty. K % 64 != 0 goes to a slower tiled kernel:
    // above two slabs with a 128 x 128 tile per CU, else above four.
    const int64_t tiles128 = ((M + 127) / 128) * ((N + 127) / 128);
    bool tiled = w8_direct_ok(K, ldx, ldw) ? M > 128 || (M > SKINNY_W8_SLAB && N * K >= (M <= 80 ? 22ll : 6ll) * 1000 * 1000)
                                           : M > 256 || (M > 128 && tiles128 >= 256);
    if (tuning().w8_tile != TUNE_UNSET) tiled = tuning().w8_tile > 0 && M > 16;
    if (tiled && N % 4 == 0 && ldy % 4 == 0 && aligned(y_dev, 8) && (!bias_dev || aligned(bias_dev, 8)) && n_out <= 256 &&
        aligned(addend_dev, 8) && ldadd % 4 == 0 && aligned(copy_dev, 8)) {
        const int rc = gemm_w8_dispatch(x_dev, wq_dev, scale_dev, outlier_idx_dev, w_out_dev, n_out, bias_dev, addend_dev, ldadd, copy, y_dev, M, N, K, ldx,
                                        ldw, ld_wout, ldy, dtype, act, s);
        if (rc != TPAMD_ERR_UNSUPPORTED) return rc;  // else no scratch memory, and the slabs need none
    }
    for (int64_t m0 = 0; m0 < M; m0 += SKINNY_W8_SLAB) {  // weights are re-streamed once per slab of 64 rows
        const int64_t mm = M - m0 < SKINNY_W8_SLAB ? M - m0 : SKINNY_W8_SLAB;
        int rc = skinny_dispatch(static_cast<const char *>(x_dev) + m0 * ldx * esz, wq_dev, nullptr, bias_dev,
                                 addend_dev ? static_cast<const char *>(addend_dev) + m0 * ldadd * esz : nullptr, ldadd, scale_dev,
                                 outlier_idx_dev, w_out_dev, n_out, static_cast<char *>(y_dev) + m0 * ldy * esz, mm, N, K, ldx,
                                 ldw, ldy, ld_wout, dtype, act, false, true, s, nullptr, copy);
        if (rc != TPAMD_OK) return rc;
    }
    return TPAMD_OK;
}

extern "C" int tpamd_linear_w8(const void *x_dev, const void *wq_dev, const void *scale_dev, const void *outlier_idx_dev,
                               const void *w_out_dev, int64_t n_out, const void *bias_dev, void *y_dev, int64_t M, int64_t N,
                               int64_t K, int64_t ldx, int64_t ldw, int64_t ld_wout, int64_t ldy, int dtype, int act,
                               void *stream) {
    return w8_entry("tpamd_linear_w8", x_dev, wq_dev, scale_dev, outlier_idx_dev, w_out_dev, n_out, bias_dev, nullptr, 0, y_dev, nullptr, M, N, K, ldx, ldw,
                    ld_wout, ldy, dtype, act, stream);
}

// As tpamd_linear_add and tpamd_linear_add_copy: the sum of two ranks' int8 Linears without a launch for the sum and one for its copy (5.0 and 4.6 us at
// 16 rows of 8192, 9.7 and 7.8 at 1024).
extern "C" int tpamd_linear_w8_add(const void *x_dev, const void *wq_dev, const void *scale_dev, const void *outlier_idx_dev, const void *w_out_dev,
                                   int64_t n_out, const void *bias_dev, const void *addend_dev, void *y_dev, void *copy_dev, int64_t M, int64_t N, int64_t K,
                                   int64_t ldx, int64_t ldw, int64_t ld_wout, int64_t ldadd, int64_t ldy, int dtype, int act, void *stream) {
    const char *who = "tpamd_linear_w8_add";
    TPAMD_REQUIRE(addend_dev != nullptr || M == 0 || N == 0, "%s: addend is NULL", who);
    TPAMD_REQUIRE(copy_dev == nullptr || copy_dev != y_dev, "%s: the copy is y", who);
    return w8_entry(who, x_dev, wq_dev, scale_dev, outlier_idx_dev, w_out_dev, n_out, bias_dev, addend_dev, ldadd, y_dev, copy_dev, M, N, K, ldx, ldw,
                    ld_wout, ldy, dtype, act, stream);
}

extern "C" int tpamd_linear_w8_ranks(int n, const tpamd_w8_rank *ranks, int64_t n_out, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw,
                                     int64_t ld_wout, int64_t ldy, int dtype, int act, void *stream) {
    const char *who = "tpamd_linear_w8_ranks";
    TPAMD_REQUIRE(n >= 0 && (n == 0 || ranks != nullptr), "%s: null pointer", who);
    for (int i = 0; i < n; ++i) {
        const tpamd_w8_rank &a = ranks[i];
        // one slab of the weight-streaming kernels; what single calls refuse or take elsewhere stays with them
        bool both = i + 1 < n && M > 0 && M <= SKINNY_W8_SLAB && N > 0 && n_out >= 0 && n_out <= K && K < (1ll << 31) && N < (1ll << 31) &&
                    (dtype == TPAMD_BF16 || dtype == TPAMD_F16) && (act == TPAMD_ACT_NONE || act == TPAMD_ACT_GELU) && K % 16 == 0 && ldw % 16 == 0 &&
                    ldx % 8 == 0 && ldx >= K && ldw >= K && ldy >= N && (n_out == 0 || ld_wout >= n_out) && tuning().w8_tile == TUNE_UNSET;
        for (int j = i; both && j < i + 2; ++j) {
            const tpamd_w8_rank &r = ranks[j];
            both = r.x && r.wq && r.scale && r.y && aligned(r.x, 16) && aligned(r.wq, 16) && (n_out == 0 || (r.outlier_idx && r.w_out)) &&
                   (r.bias == nullptr) == (a.bias == nullptr);
        }
        if (both) {
            const tpamd_w8_rank &b = ranks[i + 1];
            const bool o = n_out > 0;
            const RankStep to = {bytes_from(a.x, b.x), bytes_from(a.wq, b.wq), 0, bytes_from(a.bias, b.bias), bytes_from(a.y, b.y),
                                 bytes_from(a.scale, b.scale), o ? bytes_from(a.outlier_idx, b.outlier_idx) : 0, o ? bytes_from(a.w_out, b.w_out) : 0};
            const int rc = skinny_dispatch(a.x, a.wq, nullptr, a.bias, nullptr, 0, a.scale, a.outlier_idx, a.w_out, n_out, a.y, M, N, K, ldx, ldw, ldy,
                                           ld_wout, dtype, act, false, true, static_cast<hipStream_t>(stream), &to);
            if (rc == TPAMD_OK) ++i;
            if (rc == TPAMD_OK) continue;
            if (rc != TPAMD_ERR_UNSUPPORTED) return rc;  // else nothing was launched: too little scratch memory for two
        }
        const int rc = tpamd_linear_w8(a.x, a.wq, a.scale, a.outlier_idx, a.w_out, n_out, a.bias, a.y, M, N, K, ldx, ldw, ld_wout, ldy, dtype, act, stream);
        if (rc != TPAMD_OK) return rc;
    }
    return TPAMD_OK;
}
