// Cost models that choose between the GEMM kernels: host code, microseconds on this part.
#pragma once
#include <stdint.h>

namespace tpamd {

// No launch streams the weights of a 16-bit matrix (or gated pair) faster than 5 TB/s, which is what bounds a few rows of a wide one.
inline double stream_floor(int64_t N, int64_t K, bool swiglu) { return static_cast<double>(N) * K * (swiglu ? 4.0 : 2.0) / 5.0e6; }

// Predicted time (microseconds) of gemm_mid_kernel on the best of its tiles, and that tile: a launch, rounds of one block per CU, each with
// a fixed cost (first tiles, epilogue) and a time per K tile, shorter where the last round leaves CUs idle (the part clocks higher); 3 % more for two ranks, whose
// tiles share less in the caches.
// Non-negative least squares on relative errors over 985 shapes (65-8192 rows, 600-28000 columns, K 1024-14336, single matrices and pairs, one and two ranks), each tile forced and timed
// inside a HIP graph, those of up to 128 rows left out of the fit. Over all of them the choice among these tiles, the 256 x 256 and the 128 x 128 tiling (choose_tile) is 0.8 % off the best
// one (geometric mean; 45 by more than 5 %, at worst 27 %); with four of these tiles and models without a cost per launch and round it was 4.6 % off. Examples (us, then -> now): the pair 5504 x 4096 of two
// ranks at 512 rows 103 -> 87 (256 x 192), 16000 x 4096 of two ranks at 645 rows 188 -> 147 (224 x 192), 3072 x 4096 at 2103 rows 115 -> 91 (224 x 256: 240 tiles
// on 256 CUs), 6144 x 4096 at 4096 rows 183 -> 166 (512 tiles of 256 x 192 instead of 384 of 256 x 256), 2048 x 5120 x 1024 64 -> 54.
struct MidTile { int tmx, tnx; double launch, round, full, idle[3]; };  // idle: last round at most 1/2, at most 3/4, more of the CUs
constexpr MidTile MID_TILES[2][10] = {
    {{4, 6, 0.9, 5.1, 0.670, {0.558, 0.648, 0.666}}, {4, 8, 0.9, 5.5, 0.854, {0.700, 0.779, 0.869}}, {5, 6, 1.2, 6.1, 0.765, {0.628, 0.687, 0.754}},
     {5, 8, 1.6, 5.9, 0.999, {0.781, 0.873, 0.958}}, {6, 6, 1.6, 7.0, 0.872, {0.682, 0.750, 0.839}}, {6, 8, 0.0, 5.2, 1.225, {1.041, 1.178, 1.267}},
     {7, 6, 1.8, 7.6, 0.986, {0.760, 0.858, 0.961}}, {7, 8, 0.0, 6.6, 1.322, {1.106, 1.253, 1.311}}, {8, 6, 0.0, 7.2, 1.157, {0.987, 1.093, 1.184}},
     {8, 8, 0.5, 7.4, 1.442, {1.161, 1.303, 1.379}}},
    {{4, 6, 2.1, 3.8, 0.703, {0.568, 0.639, 0.687}}, {4, 8, 1.1, 4.9, 0.872, {0.720, 0.815, 0.877}}, {5, 6, 2.0, 5.2, 0.776, {0.631, 0.710, 0.759}},
     {5, 8, 2.2, 5.3, 1.013, {0.798, 0.884, 1.005}}, {6, 6, 2.6, 5.8, 0.890, {0.692, 0.758, 0.845}}, {6, 8, 0.3, 5.0, 1.247, {1.084, 1.253, 1.300}},
     {7, 6, 2.6, 6.4, 1.000, {0.767, 0.854, 0.958}}, {7, 8, 0.0, 6.6, 1.316, {1.136, 1.320, 1.400}}, {8, 6, 1.5, 6.1, 1.185, {1.000, 1.110, 1.171}},
     {8, 8, 0.8, 7.5, 1.436, {1.189, 1.359, 1.402}}},
};

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
        if (ranks == 2) us *= 1.03;
        if (us < best) { best = us; *tmx = t.tmx; *tnx = t.tnx; }
    }
    const double stream = stream_floor(N * ranks, 64ll * KT, swiglu);
    return M <= 128 && best < stream ? stream : best;
}

// Predicted time (microseconds) of the 128 x 128 tiling, with the K split and the number of LDS stages that give it,
// from a small cost model fitted on this part (least squares over 290 timings of 48 mid-sized shapes, then two sweeps of
// 100 shapes at 64-2048 rows with every split count and both stage counts, 1500 timings).
//  - two stages (two blocks fit a CU): a block that has its CU to itself takes 0.82 per K tile, two blocks sharing a CU
//    0.98 each (the pace of the CU's global->LDS path), 0.92 when blocks queue for several rounds of two per CU;
//  - four stages (one block per CU, three K tiles of look-ahead), in rounds of one block per CU: split launches 0.55 per
//    K tile; unsplit ones 0.60 when there is one row tile (every block streams weights nobody shares, about 27 GB/s
//    per CU), 0.42 with at most half the CUs busy and 0.55 otherwise for a single matrix, 0.62 (two row tiles) / 0.44 and
//    0.64 for the gated pair;
//  - no launch streams its weights (tiles_n column tiles of 16 KiB per K tile) faster than 5 TB/s;
//  - the partial tiles cost 4.6 + 0.39 per MB (written, read back and finished by a second launch; valid_rows = the
//    fraction of the tiles' rows that lie inside M: the others are not stored).
// Over the second sweep the choices are within 1.8 % of the best (split, stages) per shape; with two stages only they
// were 4.7 % off the best split (a single matrix 4096 x 4096 at 1024 rows: 51.5 us unsplit on two stages, 33.7 us on four).
inline double estimate128(int64_t tiles, int64_t tiles_m, int64_t tiles_n, int KT, int cus, double valid_rows, bool swiglu, int *splits,
                          bool *deep) {
    double best = 1e30;
    *splits = 1;
    *deep = false;
    const double stream = static_cast<double>(tiles_n) * KT * 16384.0 / 5.0e6;
    for (int sp = 1; sp <= 8; ++sp) {
        const int kt = (KT + sp - 1) / sp;
        if (sp > 1 && (kt < 4 || tiles * sp > 4ll * cus)) break;  // too little K per split / more than the scratch buffer holds
        const int64_t units = tiles * sp;
        const double finish = sp > 1 ? 4.6 + units * 0.065536 * valid_rows * 0.39 : 0.0;
        const double per_deep = sp > 1 ? 0.55
                                : tiles_m == 1 ? 0.60
                                : units * 2 <= cus ? (swiglu ? (tiles_m == 2 ? 0.62 : 0.44) : 0.42)
                                : (swiglu ? 0.64 : 0.55);
        const double loop_deep = static_cast<double>((units + cus - 1) / cus) * kt * per_deep;
        const double t_deep = (loop_deep > stream ? loop_deep : stream) + finish;
        if ((sp == 1 || units <= cus) && t_deep < best) { best = t_deep; *splits = sp; *deep = true; }  // split launches: one round only (measured)
        const double rounds = units <= cus ? 1.0 : static_cast<double>((units + 2 * cus - 1) / (2 * cus));
        const double per_kt = units <= cus ? 0.82 : units <= 2ll * cus ? 0.98 : 0.92;
        const double loop = rounds * kt * per_kt;
        const double t = (loop > stream ? loop : stream) + finish;
        if (t < best) { best = t; *splits = sp; *deep = false; }
    }
    return best;
}

// Two ranks' Linears and their sum in one launch and a finishing pass: 128 x 128 tiles, every rank's K in `splits` ranges. Predicted time (microseconds) of the
// best split, by the terms of estimate128.
inline double estimate_sum128(int64_t tiles, int64_t tiles_n, int KT, int cus, double valid_rows, int *splits, bool *deep) {
    double best = 1e30;
    const double stream = 2.0 * tiles_n * KT * 16384.0 / 5.0e6;
    for (int sp = 1; sp <= 4; ++sp) {
        const int kt = (KT + sp - 1) / sp;
        const int64_t units = tiles * 2 * sp;
        if ((sp > 1 && kt < 4) || units > 4ll * cus) break;
        const double finish = 4.6 + units * 0.065536 * valid_rows * 0.39;
        const double loop_deep = kt * 0.55, rounds = units <= cus ? 1.0 : static_cast<double>((units + 2 * cus - 1) / (2 * cus));
        const double t_deep = (loop_deep > stream ? loop_deep : stream) + finish;
        if (units <= cus && t_deep < best) { best = t_deep; *splits = sp; *deep = true; }
        const double loop = rounds * kt * (units <= cus ? 0.82 : units <= 2ll * cus ? 0.98 : 0.92);
        const double t = (loop > stream ? loop : stream) + finish;
        if (t < best) { best = t; *splits = sp; *deep = false; }
    }
    return best;
}

// Predicted time (microseconds) of a rank on the 256 x 256 tiling, and its K splits. The tiles run in rounds of one per CU; fitted on the same shapes (launches of more than half a round), a launch takes
// 4.7, a round 6.3, a K tile 1.42 in a full round (the part is power-limited then), 1.26 in a round that fills at most three quarters of the CUs and 1.43 in between. Split over K while all
// units fit one round: the partial tiles cost 4.5 us + 0.33 us per MB. (8192 x 8192 gated at 17 rows took 79.8 us here in four splits, predicted 57 without the floor, and 63.8 on 128 x 128.)
inline double estimate256(int64_t M, int64_t N, int KT, int cus, bool swiglu, int *splits) {
    const int64_t tiles = ((M + 255) / 256) * ((N + (swiglu ? 127 : 255)) / (swiglu ? 128 : 256));
    const double floor = stream_floor(N, 64ll * KT, swiglu), valid = static_cast<double>(M) / (((M + 255) / 256) * 256.0);
    double best = 1e30;
    *splits = 1;
    for (int sp = 1; sp <= 8; ++sp) {
        const int kt = (KT + sp - 1) / sp;
        const int64_t units = tiles * sp, full = units / cus, last = units % cus;
        if (sp > 1 && (units > cus || kt < 4)) break;
        const double loop = 4.7 + 6.3 * (full + (last > 0)) + kt * (full * 1.42 + (last == 0 ? 0.0 : last * 4 <= 3ll * cus ? 1.26 : 1.43));
        const double us = (loop > floor ? loop : floor) + (sp > 1 ? 4.5 + units * 0.262144 * valid * 0.33 : 0.0);
        if (us < best) { best = us; *splits = sp; }
    }
    return best;
}

// The prediction for the 128 x 128 tiling beside the others, above 128 rows: what the same shapes make of estimate128, whose own fit has no cost per launch. Launches of one round of blocks
// with four stages are faster than the others by it, unsplit pairs that fill more than half of the CUs most of all (2200 x 5120 at 641 rows 39.8 us; 51 on 128 x 192, predicted 57).
inline double beside_mid(double estimate128_us, int64_t M, int64_t units, int64_t tiles_m, bool deep, bool unsplit_pair, int cus) {
    if (M <= 128) return estimate128_us;
    const double per = !deep || units > cus ? 1.1 : tiles_m < 3 ? 1.05 : unsplit_pair && units * 2 > cus ? 0.8 : 0.95;
    return 2.5 + per * estimate128_us;
}
inline double beside_mid128(int64_t M, int64_t N, int KT, int cus, bool swiglu, int ranks) {
    const int64_t tiles_m = (M + 127) / 128, tiles_n = (N + (swiglu ? 63 : 127)) / (swiglu ? 64 : 128) * ranks;
    int splits = 1;
    bool deep = false;
    const double us = estimate128(tiles_m * tiles_n, tiles_m, tiles_n, KT, cus, static_cast<double>(M) / (tiles_m * 128.0), swiglu, &splits, &deep);
    return beside_mid(us, M, tiles_m * tiles_n * splits, tiles_m, deep, swiglu && splits == 1, cus);
}

// What takes a Linear or gated pair of `ranks` matrices above the weight-streaming kernels' rows: a tile of gemm_mid_kernel (tmx > 0), 256 x 256 tiles, which take two ranks in two launches
// (whole rounds of large tiles gain nothing from one), or 128 x 128 tiles.
struct TileChoice {
    int tmx, tnx;
    bool big;
    int splits256;
};
inline TileChoice choose_tile(int64_t M, int64_t N, int KT, int cus, bool swiglu, int ranks) {
    TileChoice c{0, 0, false, 1};
    const double t256 = estimate256(M, N, KT, cus, swiglu, &c.splits256) * ranks, t128 = beside_mid128(M, N, KT, cus, swiglu, ranks);
    c.big = t256 < t128;
    if (estimate_mid(M, N, KT, cus, swiglu, &c.tmx, &c.tnx, ranks) >= (c.big ? t256 : t128)) c.tmx = 0;
    return c;
}

// Whether two ranks' Linears and their sum on 128 x 128 tiles take less time than two launches, the second of which adds the first one's result. 512 rows of 4096 x 5504: 33.1 + 5.4 us twice, 59.0 +
// 5.6 in one; 645 rows, whose unsplit tiles of one rank fill the device, stay in two launches. Where the models are equal one launch was 2-3 % slower (4544 x 7168 at 513 rows, 5120 x 8192 at 468).
// Over 161 shapes of 65-1500 rows one launch takes 82, at 0.72 of the time of two (at worst 1.04); without the 256 x 256 tiling among the alternatives 8 more, at 1.004 (938 x 4096 x 14336 228 -> 272 us).
inline bool sum_predicted_faster(int64_t M, int64_t N, int KT, int cus) {
    const int64_t tiles_m = (M + 127) / 128, tiles_n = (N + 127) / 128, tiles = tiles_m * tiles_n;
    int tmx = 0, tnx = 0, splits = 0;
    bool deep = false;
    const double us = estimate_sum128(tiles, tiles_n, KT, cus, static_cast<double>(M) / (tiles_m * 128.0), &splits, &deep);
    const double once = beside_mid(us, M, tiles * 2 * splits, tiles_m, deep, false, cus);
    double other = beside_mid128(M, N, KT, cus, false, 1);
    const double mid = estimate_mid(M, N, KT, cus, false, &tmx, &tnx), big = estimate256(M, N, KT, cus, false, &splits);
    if (mid < other) other = mid;
    if (big < other) other = big;
    return once < 1.9 * other;
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

// Rows, columns and K of a row-parallel Linear whose sum over two ranks stays in two launches (tpamd_linear, then tpamd_linear_add_copy) whatever the older kernels for
// both ranks could take of it: where one launch of those measured slower, and what was not measured. Asked only where stream_kernel does not take the sum (stream_model.h), so that what stands
// here for 2 to 16 rows is for K that is no multiple of 64, little weight, and TPAMD_STREAM=0; the timings are those of the older kernels. In a HIP graph on rotated weights, one launch / two: 227 random
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
