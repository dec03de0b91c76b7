#include "skinny.h"
#include "gemm_tile.h"
#include "stream_model.h"

namespace tpamd {
namespace {

constexpr int ST_NW = 4;        // wavefronts per block
constexpr int ST_LDS_KB = 160;  // one block per CU
constexpr int ST_DEPTH = 4;     // most stages

// stream_kernel: y = act(x . w^T + bias) (+ addend), the gated pair, or the sum of two ranks' Linears, for up to 64 rows of x, on one block per CU.
// A block owns an even share of the output columns and all of K; its wavefronts take contiguous quarters of K (SUM: halves of a rank's K), 64 elements at a time,
// through a ring of stages of their own in LDS: NR weight rows (the pair: gate rows, then up rows) and XR rows of x, 128 bytes each, by loads that go straight into
// LDS and are waited for by count, so that no barrier is met before the end. Then the wavefronts' sums meet in LDS: no partial planes in memory and no second
// launch, which is what the K-split tiles pay for (4.6 us and what the planes weigh) at these row counts.
// Staged rows have no padding: piece c of row r is in slot c ^ ((r / 2) % 8), so 16 rows that follow one another are conflict-free on the 64 banks.
//
// Bound: HBM and the path from L2 into LDS, one after the other: t = 1.5 us + weights at 5.4 TB/s + x, which every CU reads whole, at 70-75 GB/s a CU (with the loads of x left
// out 4096 x 5504 a rank at 40 rows takes 21.9 of 30.1 us, with those of the weights left out 16.4). Tried and no faster: 8 wavefronts, more than 4 stages, 256 bytes of a row at a
// time, x through registers. A wavefront on a contiguous part of K is 6-12 % faster than one that takes every fourth 128 bytes. Weights are loaded past the caches' replacement (5 %).
// Where a wavefront's part of a row is 4 KiB or more, blocks start at different places in it: they otherwise ask for the same columns of all rows at one time, which
// the memory channels answer unevenly (8192 x 4096 a rank, sum, 8 rows 33.1 -> 24.6 us, 4096 x 5504 18.8 -> 17.1, 4608 x 8192 35.0 -> 28.0); below, it costs 1-7 %.
// In a HIP graph on rotated weights, both ranks in one launch, before -> now (us): Linear 6144 x 4096 at 24 / 64 rows 27.5 -> 21.1 / 29.7 -> 25.7 (K-split tiles and their finishing
// launch), 3072 x 4096 at 8 / 40 rows 11.8 -> 10.4 / 16.3 -> 15.0, the pair 5504 x 4096 at 24 / 40 rows 39.2 -> 33.6 / 40.1 -> 35.8 (128 x 128 tiles), the sum of 4096 x 2048 at 8 / 40
// rows 9.1 -> 7.9 / 14.0 -> 12.4, of 4096 x 5504 at 8 / 24 rows 20.0 -> 17.1 / 26.1 -> 22.2 (skinny_kernel, K-split tiles).
template <int DT, int MODE, bool SUM, int NR, int XR, int D>
__global__ __launch_bounds__(ST_NW * 64) void stream_kernel(SkinnyParams p) {
    constexpr int NT = (NR + 15) / 16, MT = (XR + 15) / 16, KK = 2;
    constexpr int RP = 8, PITCH = 128;  // rows per load, bytes of a staged row
    constexpr int NB = NR / RP, XB = XR / RP, L = NB + XB, STAGE = L * 1024, RING = D * STAGE;
    constexpr int WR = SUM ? ST_NW / 2 : ST_NW;  // wavefronts that share a rank's K
    constexpr int UP = MODE == SK_SWIGLU ? NR / 2 : 0;
    static_assert(NR % RP == 0 && XR % RP == 0 && UP % RP == 0, "whole loads");
    static_assert(ST_NW * RING <= ST_LDS_KB * 1024 && D >= 2 && (D - 1) * L < 64, "LDS, and the count in s_waitcnt");
    static_assert(NT * MT * 1024 <= RING, "the partial sums take the place of the stages");
    constexpr int XLAST = XR - (MT - 1) * 16;  // staged rows of the last 16 of x: the lanes of the others read these again
    static_assert(NT * 16 * PITCH <= STAGE && NB * 1024 + ((MT - 1) * 16 + XLAST) * PITCH <= STAGE && (XLAST & (XLAST - 1)) == 0, "fragments are read inside their stage");
    extern __shared__ __align__(16) char smem[];
    if constexpr (!SUM) take_rank(p);

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lq = lane >> 4, rb = lane >> 3;
    const int n0 = static_cast<int>(static_cast<int64_t>(p.N) * blockIdx.x / gridDim.x);
    const int cols = static_cast<int>(static_cast<int64_t>(p.N) * (blockIdx.x + 1) / gridDim.x) - n0;
    const int KU = p.K / 64;
    const int first = KU * (wave % WR) / WR, units = KU * (wave % WR + 1) / WR - first;

    const int skew = units >= 32 ? static_cast<int>(((blockIdx.x >> 3) * 5 + (blockIdx.x & 7) * 3 + blockIdx.z * 9) % static_cast<unsigned>(units)) : 0;
    const char *x = p.x, *w = p.w;
    if (SUM && wave >= WR) { x += p.to.x; w += p.to.w; }
    const uint32_t ldw = static_cast<uint32_t>(p.ldw) * 2, ldx = static_cast<uint32_t>(p.ldx) * 2;
    uint32_t w_off[NB], x_off[XB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int row = j * RP + rb, r = row - (MODE == SK_SWIGLU && j >= NB / 2 ? UP : 0);
        w_off[j] = static_cast<uint32_t>(r < cols ? r : cols - 1) * ldw + ((lane & 7) ^ ((row >> 1) & 7)) * 16;
    }
#pragma unroll
    for (int j = 0; j < XB; ++j) {
        const int row = j * RP + rb;
        x_off[j] = static_cast<uint32_t>(row < p.M ? row : p.M - 1) * ldx + ((lane & 7) ^ ((row >> 1) & 7)) * 16;
    }
    const uint32_t w_extent = static_cast<uint32_t>(cols - 1) * ldw + static_cast<uint32_t>(p.K) * 2;
    const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(w + static_cast<int64_t>(n0) * ldw, w_extent);
    const __amdgpu_buffer_rsrc_t w2_rsrc = MODE == SK_SWIGLU ? make_rsrc(p.w2 + static_cast<int64_t>(n0) * ldw, w_extent) : w_rsrc;
    const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(x, static_cast<uint32_t>(p.M - 1) * ldx + static_cast<uint32_t>(p.K) * 2);
    char *ring = smem + wave * RING;
    auto load = [&](int stage_off, int i) __attribute__((always_inline)) {  // unit number i of this wavefront (the last one again behind it)
        const int t = skew + (i < units ? i : units > 0 ? units - 1 : 0);
        const int u = first + (t < units || t == 0 ? t : t - units);
        unrolled<NB>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(MODE == SK_SWIGLU && j >= NB / 2 ? w2_rsrc : w_rsrc, (lds_void *)(ring + stage_off + j * 1024), 16,
                                                     static_cast<int>(w_off[j]), u * PITCH, 0, 2);
        });
        unrolled<XB>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            buffer_load16_to_lds(x_rsrc, x_off[j], u * PITCH, ring + stage_off + (NB + j) * 1024);
        });
    };

    f32x4 acc[NT][MT];
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
        for (int a = 0; a < MT; ++a) acc[b][a] = f32x4{0.f, 0.f, 0.f, 0.f};

    unrolled<D>([&](auto sc) { load(decltype(sc)::value * STAGE, decltype(sc)::value); });
    const uint32_t rd = lds_addr_of(ring) + l16 * PITCH;
    const uint32_t rd_last = lds_addr_of(ring) + (l16 & (XLAST - 1)) * PITCH;
    uint32_t kk_off[KK];
#pragma unroll
    for (int k = 0; k < KK; ++k) kk_off[k] = static_cast<uint32_t>(((k * 4 + lq) ^ (l16 >> 1)) * 16);
    int stage_off = 0;
    for (int i = 0; i < units; ++i) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * L) : "memory");
        u32x4 wq[KK][NT], xq[KK][MT];
        unrolled<KK>([&](auto hc) {
            constexpr int h = decltype(hc)::value;
            const uint32_t at = rd + stage_off + kk_off[h], at_last = rd_last + stage_off + kk_off[h];
            unrolled<NT>([&](auto bc) { wq[h][decltype(bc)::value] = lds_read16<decltype(bc)::value * 16 * PITCH>(at); });
            unrolled<MT>([&](auto ac) { xq[h][decltype(ac)::value] = lds_read16<NB * 1024 + decltype(ac)::value * 16 * PITCH>(decltype(ac)::value == MT - 1 ? at_last : at); });
        });
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        unrolled<KK>([&](auto hc) {
            constexpr int h = decltype(hc)::value;
            unrolled<NT>([&](auto bc) { already_landed(wq[h][decltype(bc)::value]); });
            unrolled<MT>([&](auto ac) { already_landed(xq[h][decltype(ac)::value]); });
        });
        load(stage_off, i + D);
#pragma unroll
        for (int h = 0; h < KK; ++h)
#pragma unroll
            for (int b = 0; b < NT; ++b)
#pragma unroll
                for (int a = 0; a < MT; ++a) acc[b][a] = mfma16<DT>(wq[h][b], xq[h][a], acc[b][a]);
        stage_off = stage_off + STAGE == RING ? 0 : stage_off + STAGE;
    }
    // every load into the stages has landed before the partial sums take their place
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
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
    for (int e = tid; e < cols * p.M; e += ST_NW * 64) {
        const int m = e / cols, n = e - m * cols;
        if constexpr (SUM) skinny_store_sum<DT>(p, total(0, WR, n, m), total(WR, ST_NW, n, m), m, n0 + n);
        else skinny_store_output<DT, MODE>(p, total(0, ST_NW, n, m), MODE == SK_SWIGLU ? total(0, ST_NW, n + UP, m) : 0.f, m, n0 + n);
    }
}

template <int DT, int MODE, bool SUM, int NR, int XR>
int launch_stream_nr(const SkinnyParams &p, int blocks, hipStream_t s) {
    constexpr int L = (NR + XR) / 8, DM = ST_LDS_KB / ST_NW / L, D = DM < ST_DEPTH ? DM : ST_DEPTH;
    if constexpr (DM < 2) {
        set_error("stream: too many rows");
        return TPAMD_ERR_UNSUPPORTED;
    } else {
        constexpr int LDS = ST_NW * D * L * 1024;
        auto kern = stream_kernel<DT, MODE, SUM, NR, XR, D>;
        static thread_local int configured_dev = -1;  // per instantiation and host thread
        int dev = 0;
        TPAMD_HIP(hipGetDevice(&dev));
        if (configured_dev != dev) {
            TPAMD_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
            configured_dev = dev;
        }
        hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(blocks), 1, p.sum ? 1 : p.ranks), dim3(ST_NW * 64), LDS, s, p);
        TPAMD_HIP(hipGetLastError());
        return TPAMD_OK;
    }
}

template <int DT, int MODE, bool SUM, int XR>
int launch_stream_xr(const SkinnyParams &p, int nr, int blocks, hipStream_t s) {
#define ST_ROWS(n) case n: return launch_stream_nr<DT, MODE, SUM, n, XR>(p, blocks, s)
    switch (nr) {
        ST_ROWS(32);
        ST_ROWS(48);
    }
    if constexpr (MODE == SK_LINEAR) {
        switch (nr) {
            ST_ROWS(16);
            ST_ROWS(24);
        }
    }
    if constexpr (!SUM) {
        switch (nr) {
            ST_ROWS(64);
            ST_ROWS(80);
            ST_ROWS(96);
        }
    }
#undef ST_ROWS
    set_error("stream: no kernel of %d rows", nr);
    return TPAMD_ERR_UNSUPPORTED;
}

template <int DT>
int launch_stream(const SkinnyParams &p, bool swiglu, int nr, int blocks, hipStream_t s) {
    auto run = [&](auto xr) {
        constexpr int XR = decltype(xr)::value;
        if (p.sum) return launch_stream_xr<DT, SK_LINEAR, true, XR>(p, nr, blocks, s);
        return swiglu ? launch_stream_xr<DT, SK_SWIGLU, false, XR>(p, nr, blocks, s) : launch_stream_xr<DT, SK_LINEAR, false, XR>(p, nr, blocks, s);
    };
    if (p.M <= 8) return run(std::integral_constant<int, 8>{});
    if (p.M <= 16) return run(std::integral_constant<int, 16>{});
    if (p.M <= 24) return run(std::integral_constant<int, 24>{});
    if (p.M <= 32) return run(std::integral_constant<int, 32>{});
    if (p.M <= 40) return run(std::integral_constant<int, 40>{});
    if (p.M <= 48) return run(std::integral_constant<int, 48>{});
    return run(std::integral_constant<int, 64>{});
}

}  // namespace

// Whether the environment names another kernel for such a launch: a choice among those that took it before, by the switches that these read at its rows. (Not those that
// choose a form of one of them: TPAMD_GEMM_W4, _STAGES, _PART_X.)
static bool other_kernel_named(int64_t M, bool swiglu) {
    const Tuning &t = tuning();
    auto set = [](int knob) { return knob != TUNE_UNSET; };
    if (set(t.skinny_cg) || set(t.skinny_resident) || (swiglu && (set(t.skinny_pair) || set(t.skinny_xlds)))) return true;
    if (M > 16) return set(t.skinny_max_m) || set(t.gemm_tile) || set(t.gemm_splitk) || set(t.gemm_splitk256);
    return M <= 3 && set(t.gemv_rows);
}

// Where stream_kernel takes a launch: whatever it can with TPAMD_STREAM=1, else where it is the faster one (stream_model.h).
bool stream_pays(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int ranks, bool swiglu, bool sum, int cus) {
    if (tuning().stream == 0 || M < 2 || M > 64 || K % 64 != 0 || K < 64 || ldx >= (1ll << 22) || ldw >= (1ll << 22) || cus < ranks) return false;
    if (tuning().stream == 1) return stream_cut(N, ranks, swiglu, sum, cus).groups > 0;
    return !other_kernel_named(M, swiglu) && stream_measured_faster(M, N, K, ranks, swiglu, sum, cus);
}

int stream_dispatch(const SkinnyParams &p, int dtype, bool swiglu, hipStream_t s) {
    int dev = 0, cus = 256;
    TPAMD_HIP(hipGetDevice(&dev));
    if (int rc = device_cus(dev, &cus); rc != TPAMD_OK) return rc;
    const StreamCut cut = stream_cut(p.N, p.sum ? 1 : p.ranks, swiglu, p.sum, cus);
    TPAMD_REQUIRE(cut.groups > 0, "stream: no cut of %d columns", p.N);
    return dtype == TPAMD_BF16 ? launch_stream<TPAMD_BF16>(p, swiglu, cut.rows, cut.blocks, s) : launch_stream<TPAMD_F16>(p, swiglu, cut.rows, cut.blocks, s);
}

}  // namespace tpamd
