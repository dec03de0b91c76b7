#include "skinny.h"
#include "gemm_tile.h"

namespace tpamd {
namespace {

constexpr int SW_NW = 4;        // wavefronts per block
constexpr int SW_LDS_KB = 160;  // one block per CU
constexpr int SW_DEPTH = 4;     // most stages

// stream_w8_kernel: y = act(x . (scale * wq)^T + x[:, outliers] . w_out^T + bias) (+ addend), or the sum of two ranks' such Linears, for up to 32 rows of x: stream_kernel
// (stream.hip) for int8 weights. A block owns an even share of the output columns and all of K; its wavefronts take contiguous quarters of K (SUM: halves of a rank's K), 128
// elements at a time, through rings of their own in LDS: 128 bytes of NR weight rows, 256 bytes of XR rows of x, loads straight into LDS that are waited for by count.
// The outlier columns are divided among a rank's wavefronts by groups of 32: the first group's indices and weights are requested in front of the ring, its x behind the ring's
// first stages, and multiplied after the last unit, when the sums have been scaled. No planes in memory and no second launch.
//
// Bound: HBM (5.2-5.9 TB/s of weights at up to 16 rows), then x from L2. Both ranks in one launch, in a HIP graph on rotated weights, before (K-split planes and their finishing launch, or
// skinny_kernel and a reduction) -> now (us): 16384 x 8192 at 8 / 16 / 32 rows 55.6 -> 47.7 / 58.7 -> 49.6 / 70.8 -> 61.6, 4608 x 8192 at 16 rows 24.1 -> 20.4, the sum of 8192 x 16384 a rank
// at 8 / 16 rows 59.2 -> 45.9 / 61.1 -> 51.8, of 8192 x 4096 at 2 / 16 rows 24.1 -> 15.5 / 21.8 -> 18.1. Blocks start at different places in a row already where a wavefront's part of it is a KiB
// (sums: 2 KiB): 16384 x 8192 at 16 rows 55.1 -> 49.6 us.
// Staged rows have no padding: piece c of a weight row is in slot c ^ ((r / 2) % 8), of a row of x in slot c ^ (r % 16): 16 rows are conflict-free on the 64 banks.
template <int DT, bool SUM, int NR, int XR, int D>
__global__ __launch_bounds__(SW_NW * 64) void stream_w8_kernel(SkinnyParams p) {
    constexpr int NT = (NR + 15) / 16, MT = (XR + 15) / 16;
    constexpr int WP = 128, XP = 256;  // bytes of a staged row of weights and of x
    constexpr int NB = NR / 8, XB = XR / 4, L = NB + XB, STAGE = L * 1024, RING = D * STAGE;
    constexpr int WR = SUM ? SW_NW / 2 : SW_NW;  // wavefronts that share a rank's K
    static_assert(NR % 8 == 0 && XR % 4 == 0, "whole loads");
    static_assert(SW_NW * RING <= SW_LDS_KB * 1024 && D >= 2 && (D - 1) * L < 64, "LDS, and the count in s_waitcnt");
    static_assert(NT * MT * 1024 <= RING, "the partial sums take the place of the stages");
    constexpr int XLAST = XR - (MT - 1) * 16;  // as in stream_kernel
    static_assert(NT * 16 * WP <= STAGE && NB * 1024 + ((MT - 1) * 16 + XLAST) * XP <= STAGE && (XLAST & (XLAST - 1)) == 0, "fragments are read inside their stage");
    extern __shared__ __align__(16) char smem[];
    if constexpr (!SUM) take_rank(p);

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lq = lane >> 4;
    const int n0 = static_cast<int>(static_cast<int64_t>(p.N) * blockIdx.x / gridDim.x);
    const int cols = static_cast<int>(static_cast<int64_t>(p.N) * (blockIdx.x + 1) / gridDim.x) - n0;
    const int KU = p.K / 128;
    const int first = KU * (wave % WR) / WR, units = KU * (wave % WR + 1) / WR - first;
    // as in stream_kernel, but for shorter parts
    const int skew = units >= (SUM ? 16 : 8) ? static_cast<int>(((blockIdx.x >> 3) * 5 + (blockIdx.x & 7) * 3 + blockIdx.z * 9) % static_cast<unsigned>(units)) : 0;

    // this wavefront's rank
    const char *x = p.x, *w = p.w, *wo = p.w_out;
    const float *scale = p.scale;
    const int *outliers = p.outlier_idx;
    if (SUM && wave >= WR) {
        x += p.to.x; w += p.to.w; wo += p.to.w_out;
        scale = reinterpret_cast<const float *>(reinterpret_cast<const char *>(scale) + p.to.scale);
        outliers = reinterpret_cast<const int *>(reinterpret_cast<const char *>(outliers) + p.to.outlier_idx);
    }

    // rows and outliers past the last ones are the last ones: rows are never stored, outliers count as zero
    float sc[NT][4];
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = b * 16 + lq * 4 + i;
            sc[b][i] = scale[n0 + (r < cols ? r : cols - 1)];
        }
    const int groups = (p.n_out + 31) / 32;
    int oi[8];
    uint32_t ow[NT][8], ox[MT][8];
    auto outlier_weights = [&](int g) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int at = g * 32 + lq * 8 + j, o = at < p.n_out ? at : p.n_out - 1;
            oi[j] = outliers[o];
#pragma unroll
            for (int b = 0; b < NT; ++b) {
                const int r = b * 16 + l16;
                ow[b][j] = reinterpret_cast<const uint16_t *>(wo)[static_cast<int64_t>(n0 + (r < cols ? r : cols - 1)) * p.ld_wout + o];
            }
        }
    };
    auto outlier_x = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int a = 0; a < MT; ++a) {
            const int m = a * 16 + l16 < p.M ? a * 16 + l16 : p.M - 1;
#pragma unroll
            for (int j = 0; j < 8; ++j) ox[a][j] = reinterpret_cast<const uint16_t *>(x)[static_cast<int64_t>(m) * p.ldx + oi[j]];
        }
    };
    const int og = wave % WR;
    if (og < groups) outlier_weights(og);

    const uint32_t ldw = static_cast<uint32_t>(p.ldw), ldx = static_cast<uint32_t>(p.ldx) * 2;
    uint32_t w_off[NB], x_off[XB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int row = j * 8 + (lane >> 3);
        w_off[j] = static_cast<uint32_t>(row < cols ? row : cols - 1) * ldw + ((lane & 7) ^ ((row >> 1) & 7)) * 16;
    }
#pragma unroll
    for (int j = 0; j < XB; ++j) {
        const int row = j * 4 + lq;
        x_off[j] = static_cast<uint32_t>(row < p.M ? row : p.M - 1) * ldx + (l16 ^ (row & 15)) * 16;
    }
    const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(w + static_cast<int64_t>(n0) * ldw, static_cast<uint32_t>(cols - 1) * ldw + static_cast<uint32_t>(p.K));
    const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(x, static_cast<uint32_t>(p.M - 1) * ldx + static_cast<uint32_t>(p.K) * 2);
    char *ring = smem + wave * RING;
    auto load = [&](int stage_off, int i) __attribute__((always_inline)) {  // unit number i of this wavefront (the last one again behind it)
        const int t = skew + (i < units ? i : units > 0 ? units - 1 : 0);
        const int u = first + (t < units || t == 0 ? t : t - units);
        unrolled<NB>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, (lds_void *)(ring + stage_off + j * 1024), 16, static_cast<int>(w_off[j]), u * WP, 0, 2);
        });
        unrolled<XB>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            buffer_load16_to_lds(x_rsrc, x_off[j], u * XP, ring + stage_off + (NB + j) * 1024);
        });
    };

    f32x4 acc[NT][MT];
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
        for (int a = 0; a < MT; ++a) acc[b][a] = f32x4{0.f, 0.f, 0.f, 0.f};

    unrolled<D>([&](auto sc_) { load(decltype(sc_)::value * STAGE, decltype(sc_)::value); });
    if (og < groups) outlier_x();
    // 16 weights of a lane, elements 64 v + 16 lq ... + 16 of a unit, meet two pieces of a row of x
    const uint32_t rd_w = lds_addr_of(ring) + l16 * WP, rd_x = lds_addr_of(ring) + NB * 1024 + l16 * XP;
    const uint32_t rd_last = lds_addr_of(ring) + NB * 1024 + (l16 & (XLAST - 1)) * XP;
    uint32_t w_at[2], x_at[4];
#pragma unroll
    for (int v = 0; v < 2; ++v) {
        w_at[v] = static_cast<uint32_t>(((v * 4 + lq) ^ (l16 >> 1)) * 16);
#pragma unroll
        for (int o = 0; o < 2; ++o) x_at[v * 2 + o] = static_cast<uint32_t>(((v * 8 + lq * 2 + o) ^ l16) * 16);
    }
    int stage_off = 0;
    for (int i = 0; i < units; ++i) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * L) : "memory");
        u32x4 wq[2][NT], xq[4][MT];
        unrolled<2>([&](auto vc) {
            constexpr int v = decltype(vc)::value;
            unrolled<NT>([&](auto bc) { wq[v][decltype(bc)::value] = lds_read16<decltype(bc)::value * 16 * WP>(rd_w + stage_off + w_at[v]); });
        });
        unrolled<4>([&](auto oc) {
            constexpr int o = decltype(oc)::value;
            unrolled<MT>([&](auto ac) { xq[o][decltype(ac)::value] = lds_read16<decltype(ac)::value * 16 * XP>((decltype(ac)::value == MT - 1 ? rd_last : rd_x) + stage_off + x_at[o]); });
        });
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        unrolled<2>([&](auto vc) { unrolled<NT>([&](auto bc) { already_landed(wq[decltype(vc)::value][decltype(bc)::value]); }); });
        unrolled<4>([&](auto oc) { unrolled<MT>([&](auto ac) { already_landed(xq[decltype(oc)::value][decltype(ac)::value]); }); });
        load(stage_off, i + D);
#pragma unroll
        for (int v = 0; v < 2; ++v)
#pragma unroll
            for (int b = 0; b < NT; ++b) {
                uint32_t q[8];
#pragma unroll
                for (int c = 0; c < 4; ++c) cvt_i8x4<DT>(wq[v][b][c], q[2 * c], q[2 * c + 1]);
#pragma unroll
                for (int o = 0; o < 2; ++o) {
                    const u32x4 half = {q[4 * o], q[4 * o + 1], q[4 * o + 2], q[4 * o + 3]};
#pragma unroll
                    for (int a = 0; a < MT; ++a) acc[b][a] = mfma16<DT>(half, xq[v * 2 + o][a], acc[b][a]);
                }
            }
        stage_off = stage_off + STAGE == RING ? 0 : stage_off + STAGE;
    }
    // every load into the stages has landed before the partial sums take their place
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
        for (int a = 0; a < MT; ++a)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[b][a][i] *= sc[b][i];
    for (int g = og; g < groups; g += WR) {
        if (g != og) {
            outlier_weights(g);
            outlier_x();
        }
        u32x4 xo[MT];
        auto packed = [&](const uint32_t (&e)[8]) __attribute__((always_inline)) {
            u32x4 q;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int at = g * 32 + lq * 8 + 2 * c;
                q[c] = (at < p.n_out ? e[2 * c] : 0u) | (at + 1 < p.n_out ? e[2 * c + 1] << 16 : 0u);
            }
            return q;
        };
#pragma unroll
        for (int a = 0; a < MT; ++a) xo[a] = packed(ox[a]);
#pragma unroll
        for (int b = 0; b < NT; ++b) {
            const u32x4 q = packed(ow[b]);
#pragma unroll
            for (int a = 0; a < MT; ++a) acc[b][a] = mfma16<DT>(q, xo[a], acc[b][a]);
        }
    }
    __syncthreads();
    f32x4 *red = reinterpret_cast<f32x4 *>(smem);
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
        for (int a = 0; a < MT; ++a) red[(wave * NT * MT + b * MT + a) * 64 + lane] = acc[b][a];
    __syncthreads();
    const float *sums = reinterpret_cast<const float *>(smem);
    auto total = [&](int from, int to, int row, int m) __attribute__((always_inline)) {
        const int at = (((row >> 4) * MT + (m >> 4)) * 64 + ((row & 15) >> 2) * 16 + (m & 15)) * 4 + (row & 3);
        float s = 0.f;
        for (int v = from; v < to; ++v) s += sums[v * NT * MT * 256 + at];
        return s;
    };
    for (int e = tid; e < cols * p.M; e += SW_NW * 64) {
        const int m = e / cols, n = e - m * cols;
        if constexpr (SUM) skinny_store_sum<DT>(p, total(0, WR, n, m), total(WR, SW_NW, n, m), m, n0 + n);
        else skinny_store_output<DT, SK_LINEAR>(p, total(0, SW_NW, n, m), 0.f, m, n0 + n);
    }
}

template <int DT, bool SUM, int NR, int XR>
int launch_stream_w8_nr(const SkinnyParams &p, int blocks, hipStream_t s) {
    constexpr int L = NR / 8 + XR / 4, DM = SW_LDS_KB / SW_NW / L, D = DM < SW_DEPTH ? DM : SW_DEPTH;
    if constexpr (DM < 2) {
        set_error("stream_w8: too many rows");
        return TPAMD_ERR_UNSUPPORTED;
    } else {
        constexpr int LDS = SW_NW * D * L * 1024;
        auto kern = stream_w8_kernel<DT, SUM, NR, XR, D>;
        static thread_local int configured_dev = -1;  // per instantiation and host thread
        int dev = 0;
        TPAMD_HIP(hipGetDevice(&dev));
        if (configured_dev != dev) {
            TPAMD_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
            configured_dev = dev;
        }
        hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(blocks), 1, SUM ? 1 : p.ranks), dim3(SW_NW * 64), LDS, s, p);
        TPAMD_HIP(hipGetLastError());
        return TPAMD_OK;
    }
}

template <int DT, bool SUM, int XR>
int launch_stream_w8_xr(const SkinnyParams &p, int nr, int blocks, hipStream_t s) {
#define SW_ROWS(n) case n: return launch_stream_w8_nr<DT, SUM, n, XR>(p, blocks, s)
    switch (nr) {
        SW_ROWS(16);
        SW_ROWS(24);
        SW_ROWS(32);
        SW_ROWS(40);
        SW_ROWS(48);
        SW_ROWS(64);
        SW_ROWS(80);
        SW_ROWS(96);
        SW_ROWS(112);
        SW_ROWS(128);
    }
#undef SW_ROWS
    set_error("stream_w8: no kernel of %d rows", nr);
    return TPAMD_ERR_UNSUPPORTED;
}

template <int DT>
int launch_stream_w8(const SkinnyParams &p, int nr, int blocks, hipStream_t s) {
    auto run = [&](auto xr) {
        constexpr int XR = decltype(xr)::value;
        return p.sum ? launch_stream_w8_xr<DT, true, XR>(p, nr, blocks, s) : launch_stream_w8_xr<DT, false, XR>(p, nr, blocks, s);
    };
    if (p.M <= 8) return run(std::integral_constant<int, 8>{});
    if (p.M <= 16) return run(std::integral_constant<int, 16>{});
    if (p.M <= 24) return run(std::integral_constant<int, 24>{});
    return run(std::integral_constant<int, 32>{});
}

}  // namespace

// How a launch of `ranks` matrices (sum: two ranks' K) would be cut: blocks of a rank and staged weight rows; false: not at all.
static bool stream_w8_cut(int64_t M, int64_t N, int ranks, bool sum, int cus, int *blocks, int *rows, int *groups) {
    const int64_t share = sum ? cus : cus / ranks;
    for (*groups = 1; *groups <= 2; ++*groups) {
        int64_t b = *groups * share;
        if (b > (N + 15) / 16) b = (N + 15) / 16;
        const int64_t cols = (N + b - 1) / b;
        for (int nr : {16, 24, 32, 40, 48, 64, 80, 96, 112, 128}) {
            if (nr < cols || nr / 8 + (M <= 8 ? 2 : M <= 16 ? 4 : M <= 24 ? 6 : 8) > SW_LDS_KB / SW_NW / 2) continue;
            *blocks = static_cast<int>(b);
            *rows = nr;
            return true;
        }
    }
    return false;
}

// Where stream_w8_kernel is the faster one. Fitted on 1386 shapes of one and of two ranks (1024-22528 columns, K 1024-16384, 2-32 rows, 0 to 96 outlier columns), timed in a HIP graph on
// rotated weights against the three kernels of pick_w8_path and their finishing pass (TPAMD_STREAM=0 and =1). Sums 0.80 of the time where it is taken or not together (the better one each time: 0.79),
// Linears 0.83 (0.82). The lines: x, which every CU reads whole, in microseconds at 70 GB/s a CU against the weights in MB (sums of 4096 x 8192 at 32 rows 27.5 -> 31.2 us, Linears of
// 1024 x 8192 13.4 -> 14.9); fewer than 2048 columns leave CUs idle (sums of 1024 x 14336 at 4 rows 1.37); 16384 columns or more of rows of one or two KiB, which no skew spreads over the
// memory channels (14336 x 1024 of two ranks at 32 rows 1.31, one 16384 x 2048 at 4 rows 1.20; rows of 1408 bytes 0.79); sums of 2048 columns, half of the CUs, on long rows (x 14336 at 4
// rows 17.2 -> 22.7 us, now 16.5). Over 2434 other shapes 0.83 of the time, 2.1 % off the better choice, 56 of them more than 3 % slower, at worst 13 %.
bool stream_w8_pays(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t n_out, int ranks, bool sum, int cus) {
    int blocks = 0, rows = 0, groups = 0;
    if (tuning().stream == 0 || M < 2 || M > 32 || K % 128 != 0 || n_out > 256 || ldx >= (1ll << 22) || ldw >= (1ll << 22) || cus < ranks) return false;
    if (!stream_w8_cut(M, N, ranks, sum, cus, &blocks, &rows, &groups)) return false;
    if (tuning().stream == 1) return true;
    if (tuning().w8_cols != TUNE_UNSET || tuning().w8_split != TUNE_UNSET || tuning().skinny_cg != TUNE_UNSET) return false;  // an explicit choice among the others
    const int64_t all = N * (sum ? 1 : ranks);
    const double mb = static_cast<double>(all) * K * (sum ? 2.0e-6 : 1.0e-6), x_us = static_cast<double>(M) * K * (sum ? 4.0 : 2.0) / 70.0e3;
    if (K < 1024 || all < 2048) return false;
    if (sum) return x_us < 2.0 + 0.08 * mb && !(N <= 2048 && K > 6144 && M >= 4);
    return x_us < 0.14 * mb && !(all >= 16384 && K <= 2048 && K % 1024 == 0);
}

int stream_w8_dispatch(const SkinnyParams &p, int dtype, hipStream_t s) {
    int dev = 0, cus = 256, blocks = 0, rows = 0, groups = 0;
    TPAMD_HIP(hipGetDevice(&dev));
    if (int rc = device_cus(dev, &cus); rc != TPAMD_OK) return rc;
    TPAMD_REQUIRE(stream_w8_cut(p.M, p.N, p.sum ? 1 : p.ranks, p.sum, cus, &blocks, &rows, &groups), "stream_w8: no cut of %d columns", p.N);
    return dtype == TPAMD_BF16 ? launch_stream_w8<TPAMD_BF16>(p, rows, blocks, s) : launch_stream_w8<TPAMD_F16>(p, rows, blocks, s);
}

}  // namespace tpamd
