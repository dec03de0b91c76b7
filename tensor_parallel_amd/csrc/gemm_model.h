// Cost models that choose between the GEMM kernels: host code, microseconds on this part.
#pragma once
#include <stdint.h>

namespace tpamd {

// No launch streams the weights of a 16-bit matrix (or gated pair) faster than 5 TB/s, which is what bounds a few rows of a wide one.
inline double stream_floor(int64_t N, int64_t K, bool swiglu) { return static_cast<double>(N) * K * (swiglu ? 4.0 : 2.0) / 5.0e6; }

// Predicted time (microseconds) of gemm_mid_kernel on the best of its tiles, and that tile: a launch, rounds of one block per CU, each with
// a fixed cost (first tiles, epilogue) and a time per K tile, shorter where the last round leaves CUs idle (the part clocks higher).
// Non-negative least squares on relative errors over 220 shapes (128-8192 rows, 1000-16000 columns, K 1024-8192, one and two ranks), each tile forced and timed
// inside a HIP graph. Over those the choice among these tiles, the 256 x 256 and the 128 x 128 tiling is 0.9 % off the best one (geometric mean); with four
// of these tiles and models of the other two tilings without a cost per launch and round it was 6.8 % off. Examples (us, before -> now): the pair 5504 x 4096 of two ranks at 512
// rows 103 -> 87 (256 x 192), at 1024 rows 177 -> 169, 16000 x 4096 of two ranks at 645 rows 188 -> 147 (224 x 192), 3072 x 4096 at 2103 rows 115 -> 91 (224 x 256: 240 tiles
// on 256 CUs), 6144 x 4096 at 4096 rows 183 -> 166 (512 tiles of 256 x 192 instead of 384 of 256 x 256), 2048 x 5120 x 1024 64 -> 54.
struct MidTile { int tmx, tnx; double launch, round, full, idle[3]; };  // idle: last round at most 1/2, at most 3/4, more of the CUs
constexpr MidTile MID_TILES[2][10] = {
    {{4, 6, 2.8, 4.7, 0.659, {0.603, 0.631, 0.662}}, {4, 8, 2.8, 5.1, 0.822, {0.737, 0.785, 0.839}}, {5, 6, 2.2, 5.5, 0.758, {0.643, 0.680, 0.774}},
     {5, 8, 3.0, 5.0, 0.989, {0.788, 0.893, 0.954}}, {6, 6, 3.4, 5.9, 0.871, {0.682, 0.745, 0.836}}, {6, 8, 2.3, 5.0, 1.154, {1.126, 1.208, 1.209}},
     {7, 6, 4.0, 6.4, 0.991, {0.755, 0.825, 0.957}}, {7, 8, 1.6, 6.7, 1.266, {1.171, 1.236, 1.287}}, {8, 6, 3.1, 6.2, 1.159, {1.058, 1.086, 1.135}},
     {8, 8, 2.2, 7.0, 1.381, {1.223, 1.256, 1.356}}},
    {{4, 6, 2.9, 3.7, 0.682, {0.616, 0.631, 0.738}}, {4, 8, 3.0, 4.9, 0.846, {0.734, 0.764, 0.817}}, {5, 6, 3.1, 4.5, 0.778, {0.644, 0.697, 0.751}},
     {5, 8, 2.5, 5.9, 0.971, {0.790, 0.871, 0.918}}, {6, 6, 2.3, 6.1, 0.866, {0.714, 0.754, 0.857}}, {6, 8, 2.9, 5.3, 1.186, {1.137, 1.199, 1.219}},
     {7, 6, 3.3, 6.3, 0.995, {0.766, 0.818, 0.907}}, {7, 8, 3.2, 5.9, 1.304, {1.160, 1.262, 1.305}}, {8, 6, 2.5, 6.9, 1.155, {1.067, 1.091, 1.191}},
     {8, 8, 3.8, 7.0, 1.411, {1.200, 1.282, 1.444}}},
};
// The prediction for the 128 x 128 tiling beside these, above 128 rows: what a fit over the same 220 shapes makes of estimate128 (gemm.hip), whose own fit has no cost per launch.
inline double beside_mid(double estimate128_us, int64_t M) { return M > 128 ? 2.5 + 1.1 * estimate128_us : estimate128_us; }

// Up to 128 rows, where nothing was fitted, at least what streaming the weights takes. Without that floor few rows of a wide matrix were
// predicted faster than HBM and taken off the 128 x 128 tiling, where a tie leaves them (us there / on these tiles): 28672 x 4096 at
// 17 / 40 / 64 / 128 rows 52 52 53 58 / 56 58 61 68, 32000 x 4096 62 62 63 62 / 65 65 67 67, the pair 14336 x 4096 52 52 53 57 / 56 56 57 60.
// Above, the floor would be wrong: 64128 x 4096 at 160 / 192 rows takes 133 / 136 us on these tiles and 142 / 144 on 256 x 256.
// `ranks`: matrices of N columns in one launch.
inline double estimate_mid(int64_t M, int64_t N, int KT, int cus, bool swiglu, int *tmx, int *tnx, int ranks = 1) {
    double best = 1e30;
    for (const MidTile &t : MID_TILES[swiglu ? 1 : 0]) {
        const int64_t bm = 32 * t.tmx, bn = (swiglu ? 16 : 32) * t.tnx;
        const int64_t tiles = ((M + bm - 1) / bm) * ((N + bn - 1) / bn) * ranks, full = tiles / cus, last = tiles % cus;
        double us = t.launch + full * (t.round + KT * t.full);
        if (last > 0) us += t.round + KT * t.idle[last * 2 <= cus ? 0 : last * 4 <= 3ll * cus ? 1 : 2];
        if (us < best) { best = us; *tmx = t.tmx; *tnx = t.tnx; }
    }
    const double stream = stream_floor(N * ranks, 64ll * KT, swiglu);
    return M <= 128 && best < stream ? stream : best;
}

// Rows, columns and K of an int8 Linear whose stream has no scratch memory (captured before its first use, or beyond the 32 buffers of a
// device): whether slabs of 64 rows through the weight-streaming kernels take it, or a tiled kernel in one K range (without outlier columns
// gemm_w8_direct_kernel, with them gemm_w8_kernel, which needs no packed ones). Predicted times, fitted to 288 timings of 18 matrices (512-65536
// columns, K 1024-16384) at 65-400 rows with 0 and 41 outlier columns on such a stream; the choice is 0.4 % off the better one (geometric mean; at
// worst 36 %, 32 us for 24). Tiles alone are 20 % off on the larger eight of them: 4096 x 5504 at 65 rows 60 us (79 with outliers) for 25 (26),
// 1024 x 16384 at 128 rows 157 (217) for 69 (70).
inline bool w8_slabs_without_scratch(int64_t M, int64_t N, int64_t K, bool outliers) {
    const double k = static_cast<double>(K) / 4096.0;
    return M / 64.0 * (5.0 + k * (5.5 + N / 512.0)) <= 6.0 + k * (outliers ? 53.0 : 36.0);
}

// Rows, columns and K of a row-parallel Linear whose sum over two ranks stays in two launches (tpamd_linear, then tpamd_linear_add_copy) whatever the kernels for
// both ranks could take of it: where one launch measured slower, and what was not measured. In a HIP graph on rotated weights, one launch / two: 227 random
// shapes of 1024-8192 columns, K 1024-8192 and 1-600 rows 0.76 (geometric mean), of which five above 1.02. Those, and what 550 more timings of longer and wider
// matrices found, are the exceptions here, by rounds of one 16-column tile per CU (a ragged count does not end on a whole round):
//  - 1 row: long rows, which the kernel for one matrix streams as fast (4096 x 8192: 24.9 us in two, 26.2 in one; ragged 5120 x 5504: 24.1, 26.8).
//  - 2 rows of at most 2048 columns beyond the row kernel's K (1024 x 8192: 13.2, 16.0; 2048 x 6144 to x 16384 0.99-1.12); of a ragged count at K up to 4096
//    (5568 x 4096: 20.4, 27.3; 4544 x 2752: 15.1, 15.8). 3 rows of those at K near 2048 (5120 x 2048 1.12, 10240 x 2048 1.33).
//  - up to 16 rows of ragged counts from 4/3 rounds and K = 4096 on (5568 and 6000 columns: x 4096 1.04-1.13, x 6144 1.00-1.07, x 8192 1.07-1.19), from 3/2 rounds and
//    K = 3072 on (7168 x 4096 at 8 rows: 25.1, 29.1).
//  - more than two rounds (8192 columns): 3 to 16 rows of ragged counts (8704-18432 columns 0.77-1.48), 9 to 16 of whole ones on K above 2048 (20480 x 6144 at 16
//    rows: 85.2, 98.7; the columns that one matrix's kernels take several tiles a block); from 17 rows on K above 2048 or more than four rounds (18432 x 4096 at 24
//    rows: 81.3, 100.5; 10240 x 8192: 76.7, 94.4), where nothing predicts which side is faster.
// With them, wider than 8192 columns 0.84 (244 timings, before 0.91 of 436 with 85 above 1.02; now 4, at most 1.04); another 229 random shapes in the first range 0.75, two above 1.02
// (1888 x 8192 at 315 rows 1.07). Left as they are: K = 6144 on 4864-5120 columns (1.00-1.13 in two runs, x 5632 and x 7168 0.87-0.97), 8192 x 28672 at 16 and 256 rows (1.10).
inline bool sum_in_two_launches(int64_t M, int64_t N, int64_t K, int cus) {
    if (K < 1024 || M < 1) return true;  // no shorter row was measured
    const int64_t tiles = (N + 15) / 16;
    const bool ragged = tiles > cus && tiles % cus != 0;
    if (M == 1) return ragged ? K > 4096 || (K > 2048 && K < 3072) : K > 11 * 512;
    if (M == 2 && (N <= 2048 ? K > 11 * 512 : ragged && K > 2048 && K <= 4096)) return true;
    if (M == 3 && ragged && K > 1536 && K <= 2048) return true;
    if (tiles > 2ll * cus) {
        if (M <= 16) return ragged ? M > 2 || K > 2048 : M > 8 && K > 2048;
        return K > 2048 || tiles > 4ll * cus;
    }
    return M <= 16 && ragged && (tiles * 2 >= 3ll * cus ? K >= 3072 : tiles * 3 >= 4ll * cus && K >= 4096);
}

// A K split count that the environment asks for, as a launch takes it: 1 to `most`, none without a K tile.
inline int forced_splits(int wanted, int KT, int most) {
    const int top = KT < most ? KT : most;
    return wanted > top ? top : wanted < 1 ? 1 : wanted;
}

}  // namespace tpamd
