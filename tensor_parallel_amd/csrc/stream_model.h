// How stream_kernel (stream.hip) cuts a launch, and where it is the faster one (host code).
#pragma once
#include <stdint.h>

namespace tpamd {

// A launch of `ranks` matrices (sum: two ranks' K): blocks of a rank, staged weight rows, and in how many turns of one block per CU it runs; groups = 0: not at all.
struct StreamCut {
    int blocks, rows, groups;
};
inline StreamCut stream_cut(int64_t N, int ranks, bool swiglu, bool sum, int cus) {
    const int64_t share = sum ? cus : cus / ranks, most = sum ? 48 : 96;
    for (int groups = 1; groups <= 4; ++groups) {
        int64_t b = groups * share;
        if (b > (N + 15) / 16) b = (N + 15) / 16;
        const int64_t cols = (N + b - 1) / b;
        int64_t nr = swiglu ? (cols + 7) / 8 * 16 : (cols + 7) / 8 * 8;
        if (nr < (swiglu ? 32 : 16)) nr = swiglu ? 32 : 16;
        if (nr > 24) nr = (nr + 15) / 16 * 16;
        if (nr <= most) return {static_cast<int>(b), static_cast<int>(nr), groups};
    }
    return {0, 0, 0};
}

// Fitted to 5717 shapes (2-64 rows, 300-28500 columns, K 1024-14336, one and two ranks), each timed in HIP graphs on weights that rotate through more memory than the caches hold, on
// stream_kernel and on the kernels that took it before. Time relative to those (geometric mean; in brackets with the better one each time):
//   rows         3             4-16          17-32         33-64
//   Linears      0.92 (0.90)   0.94 (0.93)   0.88 (0.85)   0.94 (0.91)
//   pairs        1    (0.95)   0.99 (0.96)   0.88 (0.86)   0.92 (0.89)
//   sums         0.83 (0.83)   0.86 (0.86)   0.89 (0.88)   0.97 (0.95)
// 58 of them are more than 3 % slower than there, the worst 12 %; under a rule without the exceptions marked * 257 were, up to 50 %. By rows:
//  - a sum of two ranks: 2 rows of 4096 columns or more, 3 to 16 always; above while a CU reads x in less time than K ranges of tiles need for their planes and second
//    launch. *Beyond 12288 columns at more than 32 rows only rows of whole 8 KiB (16000 x 4096 at 36 rows 75.6 -> 59.5 us; x 1408 at 64 25.3 -> 35.6), whose columns fall on few memory
//    channels in kernels that read them in step.
//  - Linears of 3 to 16 rows: up to 12288 columns of both ranks, K over 8192, and more than 8 rows on wide matrices of short rows. *3 rows: not up to 2048 columns (452 x 8192 5.8 -> 8.2)
//    nor beyond 6144 of short rows (11008 x 2048 9.6 -> 10.9), where the row kernel is faster. *Not where x weighs about as much as a CU's 16 columns (2048 x 8128 at 12 rows 11.0 -> 12.3).
//  - of 17 to 64 rows: one block per CU holds all columns (within the limit on x; *with long rows of x also not more rows than columns of a block: 3072 x 5120 at 28 rows 12.8 ->
//    14.7), or two take turns up to 32 rows (*beyond 26624 columns K from 5376 on or of whole 8 KiB: 16000 x 2688 of two ranks at 32 rows 33.2 -> 39.7). Short rows of wide matrices are left out.
//  - pairs of 4 to 16 rows: K over 8192, more than 8 on short rows that are not whole KiB. Of 17 to 64: where the columns fill the CUs (*2048 columns, which are half of them, at K from 2048 on
//    2048 x 2944 at 28 rows 9.4 -> 11.9; where x weighs more than those 2048 x 14336 at 40 30.3 -> 45.0), *not wide ones of short rows (11008 x 1024 at 36 13.0 -> 16.5); in turns only rows of
//    whole 8 KiB (8192 x 8192 of two ranks at 36 123 -> 91) or up to 24 rows of long ones (*8192 x 5120 at 40 60.9 -> 74.7), and not where staged rows would be a tenth padding.
inline bool stream_measured_faster(int64_t M, int64_t N, int64_t K, int ranks, bool swiglu, bool sum, int cus) {
    const StreamCut cut = stream_cut(N, ranks, swiglu, sum, cus);
    if (cut.groups == 0) return false;
    const int64_t all = N * (sum ? 1 : ranks), cols = (N + cut.blocks - 1) / cut.blocks * (swiglu ? 2 : 1);
    const bool full = cols * 10 >= cut.rows * 9, whole = K % 4096 == 0;
    const double mb = static_cast<double>(all) * K * (sum ? 2 : 1) * (swiglu ? 4.0e-6 : 2.0e-6);
    const double x_us = static_cast<double>(M) * K * (sum ? 4.0 : 2.0) / 70.0e3;  // one CU reading x
    if (K < 1024 || mb < 4.0) return false;
    if (sum) return M == 2 ? N >= 4096 : M <= 16 || (x_us < (full ? 3.5 : 3.0) + 0.045 * mb && (M <= 32 || N <= 12288 || whole));
    if (M < 3 || (swiglu && M < 4)) return false;
    if (swiglu) {
        if (M <= 16) return K > 8192 ? all >= 4096 : M > 8 && K < 3072 && K % 1024 != 0 && all >= 4096 && all <= 12000;
        if (all < 2048 || (all <= 2112 && K >= 2048 && M <= 32) || (x_us > 4.5 && all < 76 * M)) return false;
        if (all >= 9216 && K < (M <= 32 ? 1536 : 2048)) return false;
        return cut.groups == 1 || (cut.groups <= 3 && full && (whole || (M <= 24 && K >= (cut.groups == 2 ? 2816 : 4096))));
    }
    if (M <= 16) {
        if (M == 3 && (all <= 2048 || (K <= 2048 && all > 6144))) return false;
        if (M > 3 && ((K == 1024 && all >= 8192) || (all <= 4096 && ((K >= 4096 && M >= cols) || (K >= 5120 && M * 3 >= cols * 2))))) return false;
        if (K > 8192 && all >= 4096) return true;
        return all <= 12288 ? M <= 8 || K >= 2048 : M > 8 && K >= 1408 && K < 4096 && all >= 18432 && all <= 24576;
    }
    if (cut.groups == 1) return x_us < 3.0 + 0.04 * mb && (K >= 2048 || all <= 12288) && (x_us < 2.9 || M * 4 <= cols * (M <= 32 ? 5 : 8));
    return cut.groups == 2 && M <= 32 && K >= 2048 && (all <= 26624 || K > 5376 || whole);
}

}  // namespace tpamd
