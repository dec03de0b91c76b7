#include "gemm_tile.h"

namespace tpamd {
namespace {

// gemm_mid_kernel: y = act(x . w^T + bias) (+ addend), or the gated pair, on 32 * TMX x 32 * TNX x 64 tiles of 4 wavefronts (2 x 2, 16 * TMX
// x-rows by 16 * TNX w-rows each), one block per CU and one tile per block. For the launches whose 256 x 256 tiles leave CUs idle or a
// last round nearly empty and whose 128 x 128 tiles have too little reuse.
//
// LDS: NS stages of (BM + BN) rows of 128 bytes without padding; chunk c of row r sits in slot c ^ ((r / 2) % 8), so that 16 rows that
// follow one another are conflict-free on the 64 banks. (The padded blocks of the other kernels let two stages of most of these tiles fit
// where three do without: at 24-48 MFMAs a step, two stages leave a load too little time to land.)
// K tile g runs as two steps of TMX * TNX MFMAs, row tile by row tile. The w fragments have two register buffers, the x fragments one:
//   step A  MFMAs of k 0-31; behind the first TNX of them the reads of the w fragments of k 32-63, behind each row of MFMAs its x fragment
//   step B  MFMAs of k 32-63; after one row of them the barrier: tile g + 1 has landed (NS - 2 younger tiles in flight) and the stage of
//           tile g is read out; then the fragments of tile g + 1, and tile g + NS into the stage of tile g, spread over the MFMAs
// Bound: the matrix pipe at the clock its power leaves (1.8-2.0 GHz), the start and the epilogue of a launch, and CUs without a tile. By the SQ counters
// of 2103 rows in fp16 the pipes are busy 54 % of a launch of 242 tiles of 192 x 192 and 58 % of one of 473 gated tiles of 192 x 256 (two rounds); the
// fragment reads keep LDS busy 15-20 % of it and wavefronts wait for LDS 4-5 % of their time. A K tile of 192 x 192 takes 0.69 us
// with half of the CUs idle and 0.88 in a full round, where its MFMAs need 0.48 at 2.4 GHz; 192 x 256, on two stages, 1.04-1.25 (0.64): the fits of MID_TILES.
template <int DT, int MODE, int TMX, int TNX, int NS>
__global__ __launch_bounds__(256) void gemm_mid_kernel(GemmParams p) {
    constexpr int BM = 32 * TMX, BN = 32 * TNX, BN_OUT = MODE == MODE_SWIGLU ? BN / 2 : BN;
    constexpr int XREG = BM * 128, STAGE = (BM + BN) * 128;
    constexpr int LPT = TMX + TNX;  // global->LDS loads per wavefront and K tile
    constexpr int MF = TMX * TNX, BAR = TNX;
    static_assert(NS * STAGE <= 160 * 1024 && 4 * 16 * EP_PITCH <= NS * STAGE, "LDS");
    static_assert(BAR + TNX + TMX <= MF && TMX + TNX <= 16, "reads of a step, and their count in s_waitcnt");
    extern __shared__ __align__(16) char smem[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, lq = lane >> 4, wm = wave & 1, wn = wave >> 1;
    int tile_m, tile_n;
    tile_of_block(blockIdx.x, p.tiles_m * p.tiles_n * p.ranks, p.tiles_m, p.tiles_n * p.ranks, tile_m, tile_n);
    take_rank(p, tile_n);
    const int m0 = tile_m * BM, n0 = tile_n * BN_OUT, KT = p.K / BK;

    // ---- load addresses: rows past the end of an operand are clamped to its last one
    const int rb = lane >> 3;
    uint32_t x_off[TMX], w_off[TNX];
#pragma unroll
    for (int i = 0; i < TMX; ++i) {
        const int row = (wave * TMX + i) * 8 + rb;
        const int r = m0 + row < p.M ? row : p.M - 1 - m0;
        x_off[i] = static_cast<uint32_t>(r) * static_cast<uint32_t>(p.ldx * 2) + ((lane & 7) ^ ((row >> 1) & 7)) * 16;
    }
    const bool up = MODE == MODE_SWIGLU && wave >= 2;  // staged w rows of the pair: BN / 2 gate rows, then BN / 2 up rows
#pragma unroll
    for (int i = 0; i < TNX; ++i) {
        const int row = (wave * TNX + i) * 8 + rb, wr = up ? row - BN / 2 : row;
        const int r = n0 + wr < p.N ? wr : p.N - 1 - n0;
        w_off[i] = static_cast<uint32_t>(r) * static_cast<uint32_t>(p.ldw * 2) + ((lane & 7) ^ ((row >> 1) & 7)) * 16;
    }
    const int x_rows = p.M - m0 < BM ? p.M - m0 : BM, w_rows = p.N - n0 < BN_OUT ? p.N - n0 : BN_OUT;
    const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(p.x + static_cast<int64_t>(m0) * p.ldx * 2,
                                                    static_cast<uint32_t>(x_rows - 1) * static_cast<uint32_t>(p.ldx * 2) + static_cast<uint32_t>(p.K) * 2);
    const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc((up ? p.w2 : p.w) + static_cast<int64_t>(n0) * p.ldw * 2,
                                                    static_cast<uint32_t>(w_rows - 1) * static_cast<uint32_t>(p.ldw * 2) + static_cast<uint32_t>(p.K) * 2);
    auto load = [&](auto ic, int kt, int stage_off) {  // load number ic of K tile kt
        constexpr int i = decltype(ic)::value;
        if constexpr (i < TMX) buffer_load16_to_lds(x_rsrc, x_off[i], kt * (BK * 2), smem + stage_off + (wave * TMX + i) * 1024);
        else buffer_load16_to_lds(w_rsrc, w_off[i - TMX], kt * (BK * 2), smem + stage_off + XREG + (wave * TNX + i - TMX) * 1024);
    };

    // ---- fragment addresses
    const uint32_t smem_base = lds_addr_of(smem);
    const uint32_t x_rd = smem_base + (wm * TMX * 16 + l16) * 128;
    const uint32_t w_rd = smem_base + XREG + (wn * (MODE == MODE_SWIGLU ? TNX * 8 : TNX * 16) + l16) * 128;
    const uint32_t kk_off[2] = {static_cast<uint32_t>((lq ^ (l16 >> 1)) * 16), static_cast<uint32_t>(((4 + lq) ^ (l16 >> 1)) * 16)};

    f32x4 acc[TMX][TNX];
    u32x4 xq[TMX], wq[2][TNX];
#pragma unroll
    for (int a = 0; a < TMX; ++a)
#pragma unroll
        for (int b = 0; b < TNX; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto read_w = [&](auto hc, auto bc, uint32_t addr) {
        constexpr int h = decltype(hc)::value, b = decltype(bc)::value;
        constexpr int off = MODE == MODE_SWIGLU && b >= TNX / 2 ? (BN / 2) * 128 + (b - TNX / 2) * 2048 : b * 2048;
        wq[h][b] = lds_read16<off>(addr);
    };
    auto fence = []() { __builtin_amdgcn_sched_barrier(0); };
    const std::integral_constant<int, 0> half0{};
    const std::integral_constant<int, 1> half1{};

    // ---- first tiles
    unrolled<NS>([&](auto sc) {
        constexpr int s = decltype(sc)::value;
        const int kt = s < KT ? s : KT - 1;
        unrolled<LPT>([&](auto ic) { load(ic, kt, s * STAGE); });
    });
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 1) * LPT) : "memory");
    unrolled<TNX>([&](auto bc) { read_w(half0, bc, w_rd + kk_off[0]); });
    unrolled<TMX>([&](auto ac) { xq[decltype(ac)::value] = lds_read16<decltype(ac)::value * 2048>(x_rd + kk_off[0]); });
    fence();

    int cur = 0, nxt = STAGE;  // stage offsets of tiles g and g + 1
    for (int g = 0; g < KT; ++g) {
        {   // step A
            const uint32_t xa = x_rd + cur + kk_off[1], wa = w_rd + cur + kk_off[1];
            unrolled<MF>([&](auto mc) {
                constexpr int m = decltype(mc)::value, a = m / TNX, b = m % TNX;
                // younger than fragment a: the x fragments behind it and, from row 1 on, the w reads and a x reads of this step
                if constexpr (b == 0) {
                    reads_landed<a == 0 ? TMX - 1 : TMX - 1 + TNX>(xq[a]);
                    if constexpr (a == 0) unrolled<TNX>([&](auto bc) { already_landed(wq[0][decltype(bc)::value]); });
                    fence();
                }
                acc[a][b] = mfma16<DT>(wq[0][b], xq[a], acc[a][b]);
                fence();
                if constexpr (m < TNX) read_w(half1, std::integral_constant<int, (m < TNX ? m : 0)>{}, wa);
                if constexpr (b == TNX - 1) xq[a] = lds_read16<a * 2048>(xa);
                fence();
            });
        }
        {   // step B
            const uint32_t xa = x_rd + nxt + kk_off[0], wa = w_rd + nxt + kk_off[0];
            const int kload = g + NS < KT ? g + NS : KT - 1;  // past the end the last tile again, into a stage nobody reads any more
            unrolled<MF>([&](auto mc) {
                constexpr int m = decltype(mc)::value, a = m / TNX, b = m % TNX;
                if constexpr (m == BAR) {
                    // this wavefront has read tile g out, its part of tile g + 1 has landed; then everybody's
                    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NS - 2) * LPT) : "memory");
                    fence();
                }
                if constexpr (b == 0) {
                    if constexpr (m < BAR) reads_landed<TMX - 1 - a>(xq[a]);
                    else already_landed(xq[a]);
                    if constexpr (a == 0) unrolled<TNX>([&](auto bc) { already_landed(wq[1][decltype(bc)::value]); });
                    fence();
                }
                acc[a][b] = mfma16<DT>(wq[1][b], xq[a], acc[a][b]);
                fence();
                if constexpr (m >= BAR) {
                    if constexpr (m < BAR + TNX) read_w(half0, std::integral_constant<int, (m >= BAR && m < BAR + TNX ? m - BAR : 0)>{}, wa);
                    // x fragment r behind its last use and behind the w fragments, one per MFMA while behind
                    unrolled<TMX>([&](auto rc) {
                        constexpr int r = decltype(rc)::value, after = r * TNX + TNX - 1, turn = BAR + TNX + r;
                        if constexpr (m == (after > turn ? after : turn)) xq[r] = lds_read16<r * 2048>(xa);
                    });
                    constexpr int n = MF - BAR, l0 = (m - BAR) * LPT / n, l1 = (m + 1 - BAR) * LPT / n;
                    if constexpr (l1 > l0) load(std::integral_constant<int, l0>{}, kload, cur);
                }
                fence();
            });
        }
        cur = nxt;
        nxt = nxt + STAGE == NS * STAGE ? 0 : nxt + STAGE;
    }
    // every load and fragment read of this wavefront is done before another use of the stages and registers
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    unrolled<TMX>([&](auto ac) { reads_landed<0>(xq[decltype(ac)::value]); });
    unrolled<TNX>([&](auto bc) { reads_landed<0>(wq[0][decltype(bc)::value]); });
    // the sums stay in their accumulation registers through the loop (the gated epilogue otherwise has them copied in every K tile)
#pragma unroll
    for (int a = 0; a < TMX; ++a)
#pragma unroll
        for (int b = 0; b < TNX; ++b) asm volatile("" : "+a"(acc[a][b]));
    fence();
    drain_and_barrier();

    const bool wide = wide_stores(p);
    char *slab = smem + wave * (16 * EP_PITCH);  // the stages are read out
    const int m_wave = m0 + wm * TMX * 16;
    if constexpr (MODE == MODE_SWIGLU) {
        staged_epilogue<DT, MODE, false, TMX, TNX, 1, TNX / 2, TNX / 2>(p, acc, slab, m_wave, n0 + wn * (TNX * 8), lane, wide);
    } else {
        constexpr int GB = TNX % 4 == 0 ? 4 : TNX % 3 == 0 ? 3 : 2, GROUPS = TNX / GB;
        const int n_wave = n0 + wn * (TNX * 16);
        if (p.act == TPAMD_ACT_GELU) {
            if (p.addend != nullptr) staged_epilogue<DT, MODE, true, TMX, TNX, GROUPS, GB, 0, true>(p, acc, slab, m_wave, n_wave, lane, wide);
            else staged_epilogue<DT, MODE, true, TMX, TNX, GROUPS, GB, 0>(p, acc, slab, m_wave, n_wave, lane, wide);
        } else if (p.addend != nullptr) staged_epilogue<DT, MODE, false, TMX, TNX, GROUPS, GB, 0, true>(p, acc, slab, m_wave, n_wave, lane, wide);
        else staged_epilogue<DT, MODE, false, TMX, TNX, GROUPS, GB, 0>(p, acc, slab, m_wave, n_wave, lane, wide);
    }
}

template <int DT, int MODE, int TMX, int TNX, int NS>
int launch_mid(GemmParams p, hipStream_t s) {
    constexpr int BM = 32 * TMX, BN_OUT = MODE == MODE_SWIGLU ? 16 * TNX : 32 * TNX, LDS = NS * 32 * (TMX + TNX) * 128;
    auto kern = gemm_mid_kernel<DT, MODE, TMX, TNX, NS>;
    static thread_local int configured_dev = -1;
    int dev = 0;
    TPAMD_HIP(hipGetDevice(&dev));
    if (configured_dev != dev) {
        TPAMD_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
        configured_dev = dev;
    }
    p.tiles_m = (p.M + BM - 1) / BM;
    p.tiles_n = (p.N + BN_OUT - 1) / BN_OUT;
    const int64_t tiles = static_cast<int64_t>(p.tiles_m) * p.tiles_n * p.ranks;
    TPAMD_REQUIRE(tiles < (1ll << 31), "gemm: too many tiles");
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(tiles)), dim3(256), LDS, s, p);
    TPAMD_HIP(hipGetLastError());
    return TPAMD_OK;
}

template <int DT, int MODE>
int launch_mid_tile(const GemmParams &p, int tmx, int tnx, hipStream_t s) {
#define MID_TILE(tmx, tnx, stages) case tmx * 16 + tnx: return launch_mid<DT, MODE, tmx, tnx, stages>(p, s)
    switch (tmx * 16 + tnx) {  // three stages where they fit
        MID_TILE(4, 6, 3);
        MID_TILE(4, 8, 3);
        MID_TILE(5, 6, 3);
        MID_TILE(5, 8, 3);
        MID_TILE(6, 6, 3);
        MID_TILE(6, 8, 2);
        MID_TILE(7, 6, 3);
        MID_TILE(7, 8, 2);
        MID_TILE(8, 6, 2);
        MID_TILE(8, 8, 2);
    }
#undef MID_TILE
    set_error("gemm: no tile of %d x %d rows", 32 * tmx, 32 * tnx);
    return TPAMD_ERR_UNSUPPORTED;
}

}  // namespace

int gemm_mid(const GemmParams &p, int dtype, bool swiglu, int tmx, int tnx, hipStream_t s) {
    if (dtype == TPAMD_BF16) return swiglu ? launch_mid_tile<TPAMD_BF16, MODE_SWIGLU>(p, tmx, tnx, s) : launch_mid_tile<TPAMD_BF16, MODE_LINEAR>(p, tmx, tnx, s);
    return swiglu ? launch_mid_tile<TPAMD_F16, MODE_SWIGLU>(p, tmx, tnx, s) : launch_mid_tile<TPAMD_F16, MODE_LINEAR>(p, tmx, tnx, s);
}

}  // namespace tpamd
