// What the tiled GEMM files share: launch parameters, the tile order, global->LDS loads and fragment reads, MFMA wrappers and epilogues.
#pragma once
#include "common.h"

#include <type_traits>

namespace tpamd {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;

enum { MODE_LINEAR = 0, MODE_SWIGLU = 1 };

struct GemmParams {
    const char *x;
    const char *w;   // linear: weight; swiglu: gate weight
    const char *w2;  // swiglu: up weight
    const char *bias;
    const char *addend;  // linear: added to the rounded result (another rank's partial sum), or NULL
    char *y;
    int M, N, K;
    int64_t ldx, ldw, ldy, ldadd;  // elements
    int act;
    int tiles_m, tiles_n;
    float *ws;          // split-K: partial tiles, [split][tile][128 x rows][128 w rows] fp32
    int kt_per_split;   // split-K: K tiles (of 64) per split
    int splits;         // split-K of the 256 x 256 kernel: work units = tiles x splits
    int ranks;          // 1, or 2: a second rank's columns follow the first one's, `to` leads to its operands
    RankStep to;
    int64_t copy;       // every output is stored a second time that many bytes on (0: once)
    int sum;            // split-K of the 128 x 128 kernel: `splits` K ranges of each of two ranks, y = the sum of both rounded products
};

__device__ __forceinline__ bool wide_stores(const GemmParams &p) {  // 16 bytes each
    return ((reinterpret_cast<uintptr_t>(p.y) | static_cast<uintptr_t>(p.copy)) & 15) == 0 && p.ldy % 8 == 0;
}

// Which rank's column tile this is.
__device__ __forceinline__ void take_rank(GemmParams &p, int &tile_n) {
    if (tile_n < p.tiles_n) return;
    tile_n -= p.tiles_n;
    p.x += p.to.x; p.w += p.to.w; p.w2 += p.to.w2; p.bias += p.to.bias; p.y += p.to.y;
}

constexpr int BK = 64;            // K elements per stage (128 bytes of a row)
constexpr int LDS_ROW = 144;      // bytes per staged row: 128 + 16 pad, conflict-free for b128 reads
constexpr int GROUP_M = 4;        // tile rows per L2 reuse group

// Hardware spreads consecutive workgroup ids round-robin over the 8 XCDs (each with its own L2).
// Give every XCD one contiguous range of logical tile ids, then walk tiles in groups of GROUP_M tile
// rows so that the blocks resident on an XCD at one time share x and w tiles.
__device__ __forceinline__ void tile_of_block(int bid, int nblocks, int tiles_m, int tiles_n, int &tm, int &tn) {
    const int per = nblocks >> 3, rem = nblocks & 7;
    const int xcd = bid & 7, in_xcd = bid >> 3;
    const int logical = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + in_xcd;
    const int group_size = GROUP_M * tiles_n;
    const int g = logical / group_size;
    const int first_m = g * GROUP_M;
    const int gm = (tiles_m - first_m) < GROUP_M ? (tiles_m - first_m) : GROUP_M;
    const int in_group = logical - g * group_size;
    tm = first_m + in_group % gm;
    tn = in_group / gm;
}

typedef __attribute__((address_space(3))) void lds_void;
// Global->LDS load through a buffer descriptor: each lane's 16 bytes land at lds_base + lane * 16 (lds_base must be
// the same for the whole wavefront); address = descriptor base + per-lane 32-bit offset + wavefront-uniform
// offset, range-checked by the hardware against the descriptor's extent (a load beyond it returns zeros).
// No per-lane 64-bit address arithmetic is needed to step through K.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *base, uint32_t extent_bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, static_cast<int>(extent_bytes), 0x00020000);
}
__device__ __forceinline__ void buffer_load16_to_lds(__amdgpu_buffer_rsrc_t rsrc, uint32_t lane_off, uint32_t uniform_off, void *lds_base) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void *)lds_base, 16, static_cast<int>(lane_off), static_cast<int>(uniform_off), 0, 0);
}
// Fragment read that the compiler does not see as an LDS access. With ordinary loads it waits for every
// in-flight global->LDS load before each LDS read (it cannot tell that they go to the other stage), which
// serialises the pipeline; this way the waits are the counted ones written out in the main loop.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <int OFFSET>
__device__ __forceinline__ u32x4 lds_read16(uint32_t lds_addr) {
    static_assert(OFFSET >= 0 && OFFSET < 65536, "ds offset field is 16 bits");
    u32x4 v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(lds_addr), "n"(OFFSET));
    return v;
}
__device__ __forceinline__ uint32_t lds_addr_of(const void *p) {
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) char *)p));
}
// All of this wavefront's loads and LDS accesses done, then the workgroup barrier. The memory clobber keeps
// the compiler from moving LDS accesses across it.
__device__ __forceinline__ void drain_and_barrier() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

typedef __attribute__((ext_vector_type(4))) float f32x4;
template <int DT>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (DT == TPAMD_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Four consecutive output columns n..n+3 of one row, from fp32 sums to the packed 16-bit store value.
// linear: v = bias/activation of g; swiglu: g = gate sums, u = up sums.
template <int DT, int MODE>
__device__ __forceinline__ uint2 finish4(const GemmParams &p, const float (&g)[4], const float (&u)[4], int n, const char *add_row = nullptr) {
    uint2 o;
    if constexpr (MODE == MODE_SWIGLU) {
        // gate and up products rounded to the tensor dtype, then silu and the product each rounded again
        uint32_t out[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint32_t g2 = pack2_half<DT>(g[2 * j], g[2 * j + 1]);
            const uint32_t u2 = pack2_half<DT>(u[2 * j], u[2 * j + 1]);
            const uint32_t s2 = pack2_half<DT>(silu_f32(lo_half_to_f32<DT>(g2)), silu_f32(hi_half_to_f32<DT>(g2)));
            out[j] = pack2_half<DT>(lo_half_to_f32<DT>(s2) * lo_half_to_f32<DT>(u2), hi_half_to_f32<DT>(s2) * hi_half_to_f32<DT>(u2));
        }
        o.x = out[0];
        o.y = out[1];
    } else {
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = g[j];
        if (p.bias) {
            const uint2 braw = *reinterpret_cast<const uint2 *>(p.bias + static_cast<int64_t>(n) * 2);
            v[0] += lo_half_to_f32<DT>(braw.x); v[1] += hi_half_to_f32<DT>(braw.x);
            v[2] += lo_half_to_f32<DT>(braw.y); v[3] += hi_half_to_f32<DT>(braw.y);
        }
        if (p.act == TPAMD_ACT_GELU) {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = gelu_erf(v[j]);
        }
        o.x = pack2_half<DT>(v[0], v[1]);
        o.y = pack2_half<DT>(v[2], v[3]);
        if (add_row != nullptr) {  // the row of p.addend this output row belongs to
            const uint2 araw = *reinterpret_cast<const uint2 *>(add_row + static_cast<int64_t>(n) * 2);
            o.x = add_packed2<DT>(o.x, araw.x);
            o.y = add_packed2<DT>(o.y, araw.y);
        }
    }
    return o;
}

// Epilogue of the direct kernels. With w as the first MFMA operand a lane holds D[n = 4*(lane/16) + i][m = lane%16],
// i = 0..3: four consecutive output columns of one output row, one 8-byte store.
// acc[a][b]: a = 16-row tile of x (TMX per wavefront), b = 16-row tile of w (4 per wavefront; swiglu: 2 gate + 2 up).
template <int DT, int MODE, int TMX>
__device__ __forceinline__ void epilogue16(const GemmParams &p, f32x4 (&acc)[TMX][4], int m_wave, int n_wave, int l16, int lq) {
#pragma unroll
    for (int a = 0; a < TMX; ++a) {
        const int m = m_wave + a * 16 + l16;
        if (m >= p.M) continue;
        char *yrow = p.y + static_cast<int64_t>(m) * p.ldy * 2;
#pragma unroll
        for (int b = 0; b < (MODE == MODE_SWIGLU ? 2 : 4); ++b) {
            const int n = n_wave + b * 16 + lq * 4;
            if (n >= p.N) continue;  // N is a multiple of 4: the group of 4 is all in or all out
            float g[4], u[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                g[j] = acc[a][b][j];
                u[j] = MODE == MODE_SWIGLU ? acc[a][(b + 2) & 3][j] : 0.f;
            }
            const char *add_row = MODE == MODE_LINEAR && p.addend != nullptr ? p.addend + static_cast<int64_t>(m) * p.ldadd * 2 : nullptr;
            const uint2 o = finish4<DT, MODE>(p, g, u, n, add_row);
            *reinterpret_cast<uint2 *>(yrow + static_cast<int64_t>(n) * 2) = o;
            if (p.copy) *reinterpret_cast<uint2 *>(yrow + static_cast<int64_t>(n) * 2 + p.copy) = o;
        }
    }
}

// Epilogue of the 4-wavefront kernels. A lane holds 4 consecutive columns of one row per accumulator tile; stored like
// that, an instruction would write 32-byte pieces of 16 rows. Instead the packed results of 16 rows x (16 * GB)
// columns go through a wavefront-private LDS slab (16 rows, EP_PITCH bytes apart) and leave as 16 bytes per lane:
// whole 128-byte lines, 8 rows per store instruction, when GB = 4.
// acc[a][b]: a = 16-row tile of x, b = 16-row tile of w. The wavefront's columns are GROUPS runs of 16 * GB; gated pair:
// tile b holds gate sums and tile b + UP the up sums of the same columns. wide: 16-byte stores are aligned.
constexpr int EP_PITCH = 144;
// ADD: the addend (p.addend, not NULL) of the 16 rows after next is requested while the current 16 rows are converted and
// stored, one set of registers ahead: asked for at the point of use, every piece is a full memory round trip with
// nothing else to do on this SIMD (10 us on the 4096 x 4096 x 5504 down projection).
template <int DT, int MODE, bool GELU, int TMX, int NBT, int GROUPS, int GB, int UP, bool ADD = false>
__device__ __forceinline__ void staged_epilogue(const GemmParams &p, f32x4 (&acc)[TMX][NBT], char *slab, int m_wave, int n_wave,
                                                int lane, bool wide) {
    static_assert(GB >= 2 && GB <= 4, "32, 48 or 64 columns per slab");
    const int l16 = lane & 15, lq = lane >> 4;
    uint2 braw[GROUPS * GB];
    if constexpr (MODE == MODE_LINEAR) {
#pragma unroll
        for (int b = 0; b < GROUPS * GB; ++b) {
            const int n = n_wave + b * 16 + lq * 4;
            braw[b] = p.bias != nullptr && n < p.N ? *reinterpret_cast<const uint2 *>(p.bias + static_cast<int64_t>(n) * 2) : make_uint2(0, 0);
        }
    }
    constexpr int LANES_PER_ROW = GB * 2;            // 16 bytes per lane
    constexpr int READS = (16 * LANES_PER_ROW + 63) / 64;  // 48 columns: the second read has work for half the lanes
    int rd_row[READS], rd_col[READS];
#pragma unroll
    for (int h = 0; h < READS; ++h) {
        rd_row[h] = (lane + 64 * h) / LANES_PER_ROW;
        rd_col[h] = (lane + 64 * h) % LANES_PER_ROW;
    }
    uint2 addv[2][ADD ? GROUPS * READS : 1][2];
    auto request_addend = [&](int a) {
#pragma unroll
        for (int gq = 0; gq < GROUPS; ++gq)
#pragma unroll
            for (int h = 0; h < READS; ++h) {
                const int m = m_wave + a * 16 + rd_row[h];
                const int n = n_wave + gq * (16 * GB) + rd_col[h] * 8;
                const bool in = m < p.M && n < p.N && (GB != 3 || rd_row[h] < 16);
                const char *ap = p.addend + (in ? (static_cast<int64_t>(m) * p.ldadd + n) * 2 : 0);
                addv[a & 1][gq * READS + h][0] = *reinterpret_cast<const uint2 *>(ap);
                addv[a & 1][gq * READS + h][1] = in && n + 8 <= p.N ? *reinterpret_cast<const uint2 *>(ap + 8) : make_uint2(0, 0);
            }
    };
    if constexpr (ADD) request_addend(0);
#pragma unroll
    for (int a = 0; a < TMX; ++a) {
        if constexpr (ADD) {
            if (a + 1 < TMX) request_addend(a + 1);
        }
#pragma unroll
        for (int gq = 0; gq < GROUPS; ++gq) {
#pragma unroll
            for (int bb = 0; bb < GB; ++bb) {
                const int b = gq * GB + bb;
                uint2 o;
                if constexpr (MODE == MODE_SWIGLU) {
                    float gsum[4], usum[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        gsum[j] = acc[a][b][j];
                        usum[j] = acc[a][b + UP][j];
                    }
                    o = finish4<DT, MODE>(p, gsum, usum, 0);
                } else {
                    float v[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] = acc[a][b][j];
                    v[0] += lo_half_to_f32<DT>(braw[b].x); v[1] += hi_half_to_f32<DT>(braw[b].x);
                    v[2] += lo_half_to_f32<DT>(braw[b].y); v[3] += hi_half_to_f32<DT>(braw[b].y);
                    if constexpr (GELU) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) v[j] = gelu_erf(v[j]);
                    }
                    o.x = pack2_half<DT>(v[0], v[1]);
                    o.y = pack2_half<DT>(v[2], v[3]);
                }
                *reinterpret_cast<uint2 *>(slab + l16 * EP_PITCH + bb * 32 + lq * 8) = o;
            }
            __builtin_amdgcn_wave_barrier();
            asm volatile("" ::: "memory");
#pragma unroll
            for (int h = 0; h < READS; ++h) {
                const int row = rd_row[h];
                const uint4 vs = *reinterpret_cast<const uint4 *>(slab + (GB == 3 ? row & 15 : row) * EP_PITCH + rd_col[h] * 16);
                const int m = m_wave + a * 16 + row;
                const int n = n_wave + gq * (16 * GB) + rd_col[h] * 8;
                if (m >= p.M || n >= p.N || (GB == 3 && row >= 16)) continue;
                char *dst = p.y + (static_cast<int64_t>(m) * p.ldy + n) * 2;
                uint4 v = vs;
                if constexpr (ADD) {
                    {  // the lane that stores 8 outputs adds the same 8 elements of the addend
                        const uint2 a0 = addv[a & 1][gq * READS + h][0], a1 = addv[a & 1][gq * READS + h][1];
                        v.x = add_packed2<DT>(v.x, a0.x); v.y = add_packed2<DT>(v.y, a0.y);
                        v.z = add_packed2<DT>(v.z, a1.x); v.w = add_packed2<DT>(v.w, a1.y);
                    }
                }
                auto put = [&](char *to) {
                    if (n + 8 <= p.N) {
                        if (wide) *reinterpret_cast<uint4 *>(to) = v;
                        else {
                            *reinterpret_cast<uint2 *>(to) = make_uint2(v.x, v.y);
                            *reinterpret_cast<uint2 *>(to + 8) = make_uint2(v.z, v.w);
                        }
                    } else {
                        *reinterpret_cast<uint2 *>(to) = make_uint2(v.x, v.y);  // N is a multiple of 4
                    }
                };
                put(dst);
                if constexpr (MODE == MODE_LINEAR) {
                    if (p.copy) put(dst + p.copy);
                }
            }
            __builtin_amdgcn_wave_barrier();
            asm volatile("" ::: "memory");
        }
    }
}

template <int N, int I = 0, class F>
__device__ __forceinline__ void unrolled(F &&f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        unrolled<N, I + 1>(f);
    }
}

// All but the YOUNGER last LDS reads of this wavefront have arrived, the named registers among them (the reads are asm
// statements: the waits are ours).
template <int YOUNGER>
__device__ __forceinline__ void reads_landed(u32x4 &r) {
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(r) : "n"(YOUNGER) : "memory");
}
__device__ __forceinline__ void already_landed(u32x4 &r) { asm volatile("" : "+v"(r)); }  // uses stay behind the wait in front of this
template <int YOUNGER>
__device__ __forceinline__ void reads_landed(u32x4 (&r)[4]) {
    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]) : "n"(YOUNGER) : "memory");
}

// gemm_mid.hip: one launch on tiles of 32 * tmx x-rows by 32 * tnx w-rows (the gated pair: 16 * tnx columns). K a multiple of 64, leading
// dimensions below 2^22, 16-byte aligned operands with N a multiple of 4.
int gemm_mid(const GemmParams &p, int dtype, bool swiglu, int tmx, int tnx, hipStream_t s);

}  // namespace tpamd
