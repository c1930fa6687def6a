// Per-block (bm x bk, bm/bk in {32, 128}) block-scaled cast to E4M3 / E2M1 for gfx950.
//
// A workgroup owns one tile of 128 rows x TW columns (TW = 128 or 256 with 512 threads, 256 or 512 with 1024 threads: see the
// table at the launch code), i.e. 1 to 64 scale blocks.  With TW = 128, thread (t, c) = (tid / 16, tid % 16) holds
// the 8 elements at columns 8c.. of rows t, t+32, t+64, t+96: four 16-byte streaming loads per thread (bf16), all
// issued up front; the tile stays in registers between the amax reduction and the conversion, so HBM is read once.  The amax of a block is
// reduced over the bk/8 lanes that share it with DPP, then across row slots and waves through one
// LDS exchange (a partial per 16-lane row, one barrier, vector reads).
//
// Reference semantics: tile_kernels/quant/per_block_cast_kernel.py:52-136.
#include <type_traits>

#include "tk_device.hpp"
#include "tk_host.hpp"

namespace tk {

constexpr int kBlockTile = 128;
constexpr int kPerBlockThreads = 512, kMidTile = 256, kWideTile = 512, kWideThreads = 1024;   // the tile shapes: see the table at the launch code

struct PerBlockParams {
    const void *x;
    uint8_t *out;
    SfRef sf;
    int M, K;
    int tiles_m, tiles_k;
    int round_sf, mode;
};

// Parameters travel as individual scalars (16 dwords in all) so that they are preloaded into SGPRs
// at wave start (the library is built with -amdgpu-kernarg-preload-count=16).
#define TK_PB_KERNEL_ARGS                                                                                  \
    const void *a_x, uint8_t *a_out, void *a_sf, int64_t a_sf_ld, int a_M, int a_K, int a_tiles_m, int a_tiles_k, \
        int a_round_sf, int a_mode, int a_sf_layout, int a_nm, int a_nk
#define TK_PB_KERNEL_UNPACK \
    const PerBlockParams p{a_x, a_out, SfRef{a_sf, a_sf_ld, a_sf_layout, a_nm, a_nk}, a_M, a_K, a_tiles_m, a_tiles_k, a_round_sf, a_mode}
#define TK_PB_LAUNCH_ARGS(p) \
    (p).x, (p).out, (p).sf.base, (p).sf.ld, (p).M, (p).K, (p).tiles_m, (p).tiles_k, (p).round_sf, (p).mode, (p).sf.layout, (p).sf.nm, (p).sf.nk

// TW: columns of a tile (128, 256 or 512); a tile is 128 rows x TW columns.
// THREADS: threads per tile.
// FULL: the tile lies wholly inside the matrix, so no bounds checks are compiled in.
// FULL_GRID: so do all tiles of the launch.
// FEW: of a matrix of few rows, see the launch code.
template <typename InT, int FMT, int BM, int BK, int TW, int THREADS, bool FULL, bool FULL_GRID, bool FEW = false>
__device__ __forceinline__ void per_block_cast_tile(const PerBlockParams &p, uint8_t *xchg) {
    constexpr int LPR = TW / 8;                                      // lanes along a row of the tile
    constexpr int SUBM = kBlockTile / BM, SUBK = TW / BK;            // scale blocks per tile
    constexpr int LPG = BK / 8;                                      // lanes sharing a block in one row
    constexpr int TR = THREADS / LPR;                                // rows covered by one pass of the workgroup
    constexpr int NI = kBlockTile / TR;                              // rows per thread
    constexpr int IPB = BM / TR;                                     // of which per scale block
    static_assert(IPB >= 1, "a pass of the workgroup must not span two scale blocks");
    // partial maxima: one per (scale block, 16-row slot of the workgroup); no atomics, no zeroing
    __shared__ __attribute__((aligned(16))) uint32_t part[SUBM][SUBK][TR];

    const int tile_m = blockIdx.y, tile_k = blockIdx.x;   // 2-D grid: no division on the way to the first load

    const int t = threadIdx.x / LPR, c = threadIdx.x % LPR;
    const int col = tile_k * TW + c * 8;
    const int bj = (c * 8) / BK;
    const bool col_ok = FULL || col < p.K;
    const int row0 = tile_m * kBlockTile + t;
    const InT *x = reinterpret_cast<const InT *>(p.x) + (int64_t)row0 * p.K + col;
    const int64_t out_ld = FMT == TK_E4M3 ? p.K : p.K / 2;

    // fp32 input: the LPR lanes of a tile row read its 32 * LPR bytes as two whole-line loads and deal them out through LDS
    constexpr int XB = FEW ? 0 : Raw8<InT>::kXchgBytes;
    constexpr int RUN = LPR < 64 ? LPR : 64;     // lanes of one run: a tile row, or the part of it that one wave holds
    Raw8<InT> raw[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        if constexpr (FULL) {
            raw[i].template load_run<RUN>(x + (int64_t)(TR * i) * p.K, c % RUN);
        } else if constexpr (FEW) {
            raw[i].load(x + (int64_t)(TR * i) * p.K, col_ok && row0 + TR * i < p.M);
        } else {
            // No lane branches around its load: all loads of a lane go out together, where each one in a branch of its own is waited
            // for before the next (the tiles at the lower edge then end the launch some 5 us after the others).  A lane beyond the
            // last row reads that row, one beyond the last column the last columns (fp32: nothing, it is cleared): no maximum changes.
            const InT *xr = reinterpret_cast<const InT *>(p.x) + (int64_t)min(row0 + TR * i, p.M - 1) * p.K;
            if constexpr (XB != 0) {
                const int first = col - (c % RUN) * 8;
                raw[i].template load_run_part<RUN>(xr + first, c % RUN, p.K - first, p.x);
            } else {
                raw[i].load(xr + (col_ok ? col : p.K - 8));
            }
        }
        if (i + 1 < NI) vmem_issue_gap();
    }
    if constexpr (XB != 0) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            raw[i].template settle<RUN>(xchg + (threadIdx.x / RUN) * (RUN * XB), c % RUN);
            if (!col_ok) raw[i].zero();
        }
    }

    float inv[SUBM];
    if (p.mode != TK_CAST_GIVEN_SF) {
#pragma unroll
        for (int b = 0; b < SUBM; ++b) {
            float m = 0.0f;
#pragma unroll
            for (int i = b * IPB; i < (b + 1) * IPB; ++i) {
                float v[8];
                raw[i].get(v);
                m = __builtin_fmaxf(m, absmax8(v));
            }
            m = group_allmax<LPG>(m);
            if ((c % LPG) == 0) part[b][bj][t] = f2u(m);
        }
        __syncthreads();
#pragma unroll
        for (int b = 0; b < SUBM; ++b) {
            uint32_t m = 0;
#pragma unroll
            for (int q = 0; q < TR; q += 4) {
                const u32x4 w = *reinterpret_cast<const u32x4 *>(&part[b][bj][q]);
                m = umax(umax(m, umax(w.x, w.y)), umax(w.z, w.w));
            }
            const Scale sc = make_scale<Fmt<FMT>::qmax>(u2f(m), Fmt<FMT>::floor_, p.round_sf != 0);
            inv[b] = sc.inv;
            // one thread per scale block stores it: the first row slot's first lane of the block
            if (t == 0 && (c % LPG) == 0) {
                const int mb = tile_m * SUBM + b, kb = tile_k * SUBK + bj;
                if (mb < p.sf.nm && kb < p.sf.nk) sf_store(p.sf, mb, kb, sc);
            }
        }
    } else {
#pragma unroll
        for (int b = 0; b < SUBM; ++b) {
            const int m = tile_m * SUBM + b, k = tile_k * SUBK + bj;
            const float s = (m < p.sf.nm && k < p.sf.nk) ? sf_load(p.sf, m, k) : 1.0f;
            inv[b] = 1.0f / s;
        }
    }
    if (p.mode == TK_SF_ONLY) return;

    // The two lanes that hold 16 neighbouring columns exchange the codes of two row slots, so that each stores 16 consecutive codes of
    // one row with one instruction: half as many store instructions, each twice as wide.  A launch of wide tiles fits the GPU in one
    // round, all its workgroups finish loading at about the same time (measured: the last load of every workgroup of [7168, 2048]
    // arrives between 3.4 and 4.7 us after the start) and the rest of the launch is one burst of stores, which drains faster in fewer,
    // wider instructions: bf16 [7168, 2048] -> E4M3 8.54 -> 8.20 us, [4096, 4096] 9.22 -> 8.66, [8192, 2048] 9.94 -> 9.07.
    // (128-column tiles gain to E2M1 where the matrix is ragged, bf16 [3666, 576] 3.38 -> 3.09, [7830, 960] 6.0 -> 5.5; not where all tiles
    // are whole, [1536, 2048] 2.92 -> 3.23, nor fp32, [2560, 2048] 6.45 -> 6.54, nor, of more than some 1000 tiles, E4M3, whose workgroups
    // finish loading at different times so that loads and stores overlap: [3589, 6144] 12.54 -> 12.75.)
    constexpr bool PAIRED = !FEW && NI % 2 == 0 && (TW > kBlockTile || (!FULL_GRID && FMT == TK_E2M1 && std::is_same<InT, bf16_t>::value));
    if constexpr (PAIRED) {
        const bool odd = threadIdx.x & 1;
#pragma unroll
        for (int i = 0; i < NI; i += 2) {
            float v[8];
            raw[i].get(v);
            const u32x2 a = p.mode == TK_CAST_GIVEN_SF ? quantise8<FMT, true>(v, inv[i / IPB]) : quantise8<FMT, false>(v, inv[i / IPB]);
            raw[i + 1].get(v);
            const u32x2 b = p.mode == TK_CAST_GIVEN_SF ? quantise8<FMT, true>(v, inv[(i + 1) / IPB]) : quantise8<FMT, false>(v, inv[(i + 1) / IPB]);
            // the even lane keeps slot i and takes its neighbour's half of it, the odd lane likewise with slot i + 1
            const u32x2 send = odd ? a : b;
            const u32x2 recv = {dpp_u32<kDppXor1>(send.x), FMT == TK_E4M3 ? dpp_u32<kDppXor1>(send.y) : 0u};
            const u32x2 lo = odd ? recv : a, hi = odd ? b : recv;
            const int row = row0 + TR * (i + (odd ? 1 : 0));
            if (!FULL && (!col_ok || row >= p.M)) continue;      // (K is a multiple of 64: both lanes have columns, or neither)
            uint8_t *out_row = p.out + (int64_t)row * out_ld;
            if (FMT == TK_E4M3) st_stream16(out_row + (col & ~15), u32x4{lo.x, lo.y, hi.x, hi.y});
            else st_stream8(out_row + ((col & ~15) >> 1), u32x2{lo.x, hi.x});
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int row = row0 + TR * i;
        if (FULL || (col_ok && row < p.M)) {
            float v[8];
            raw[i].get(v);
            uint8_t *out_row = p.out + (int64_t)row * out_ld;
            if (p.mode == TK_CAST_GIVEN_SF) quantise_store8<FMT, true>(v, inv[i / IPB], out_row, col);
            else quantise_store8<FMT, false>(v, inv[i / IPB], out_row, col);
        }
    }
}

// FULL_GRID: M and K are multiples of 128.  Otherwise only the tiles on the lower and right edges take the
// bounds-checked path; the choice is uniform over the workgroup.  (With every tile checked, bf16 [32767, 4096] took
// 63.9 us against 59.1 us for [32768, 4096].)
template <typename InT, int FMT, int BM, int BK, int TW, int THREADS, bool FULL_GRID, bool FEW = false>
__global__ __launch_bounds__(THREADS) void per_block_cast_kernel(TK_PB_KERNEL_ARGS) {
    TK_PB_KERNEL_UNPACK;
    constexpr int XB = FEW ? 0 : Raw8<InT>::kXchgBytes;
    __shared__ __attribute__((aligned(16))) uint8_t xchg[XB ? THREADS * XB : 16];      // (one for both kinds of tile)
    if constexpr (FULL_GRID) {
        per_block_cast_tile<InT, FMT, BM, BK, TW, THREADS, true, true>(p, xchg);
    } else if constexpr (FEW) {
        per_block_cast_tile<InT, FMT, BM, BK, TW, THREADS, false, false, true>(p, xchg);
    } else {
        if (((int)blockIdx.y + 1) * kBlockTile <= p.M && ((int)blockIdx.x + 1) * TW <= p.K)
            per_block_cast_tile<InT, FMT, BM, BK, TW, THREADS, true, false>(p, xchg);
        else
            per_block_cast_tile<InT, FMT, BM, BK, TW, THREADS, false, false>(p, xchg);
    }
}

// Tile shapes, measured on MI355X for bf16 -> E4M3 128x128 (us per call):
//                                          [2048,2048]  [7168,2048]  [4096,4096]  [4096,7168]  [8192,4096]  [16384,7168]
//   128 x 128, 512 threads (4 rows/thread)     4.07         9.13        10.02        15.58        17.46        52.1
//   128 x 512, 1024 threads (8 rows/thread)    6.02         8.60         9.19        16.36        18.45
//   128 x 512, 512 threads (16 rows/thread)    6.31         8.87         9.82        16.59        20.37        58.8
//   128 x 256, 1024 threads                    4.72         9.30        10.57        16.39        18.06
// (128 x 128 with 256 threads: 9.4 at [7168,2048], with 1024: 9.8.)  A wave of a 512-column tile reads 1 KB of one
// row per load instruction instead of 256 bytes of four rows.  Its workgroup of 1024 threads at 96 registers has a CU to itself, so
// that the launch is as long as the CU with the most tiles: the wide tile pays where there are at most 256 of them and not much fewer
// than 140, and 256 columns with 1024 threads where there are at most 256 of those and not fewer than 192, to E4M3 from fp32 150.  us, 128 / 256
// (1024 threads) / 512 columns:
//   E4M3 bf16 [3072,2048] 4.85 / 4.79 / 6.30, [3584,2048] 5.30 / 4.97 / 6.50, [4096,2048] 5.66 / 5.22 / 6.62, [2100,4096] 5.94 / 6.46 / 6.47,
//   [4608,2048] 6.78 / 7.61 / 6.75, [6144,2048] 7.82 / 8.33 / 7.44, [7168,2048] 8.90 / 9.17 / 8.29, [8192,2048] 9.74 / 10.12 / 9.23, [8704,2048]
//   10.79 / 11.83 / 11.93, [9044,2048] 11.0 / 12.1 / 13.3, [4100,4096] 9.90 / 10.5 / 10.8, [5000,4096] 11.9 / 12.5 / 13.75
//   fp32 [2560,2048] 6.39 / 6.17 / 8.38, [4096,2048] 8.39 / 7.61 / 9.03, [4608,2048] 9.74 / 10.90 / 9.30, [8192,2048] 14.98 / 15.22 / 13.98,
//   [9044,2048] 16.5 / 18.4 / 20.0
// To E2M1 the wide tile begins to pay later, from 160 of them for bf16 and 208 for fp32 (there for two widths of three):
//   bf16 [3072,2048] 4.63 / 4.55 / 5.99, [3584,2048] 5.35 / 4.84 / 6.57, [4096,2048] 5.54 / 5.08 / 6.76, [2304,4096] 6.52 / 6.60 / 6.47, [4608,2048] 6.58 / 6.67 /
//   6.91, [5376,2048] 7.16 / 6.97 / 6.91, [2688,4096] 7.16 / 7.02 / 6.70, [7168,2048] 8.80 / 7.82 / 7.76, [8192,2048] 9.14 / 8.60 / 8.77, [4096,4096] 9.22 / 8.73 / 8.03
//   fp32 [1408,4096] 6.83 / 6.97 / 8.98, [3072,2048] 6.51 / 6.49 / 8.76, [3584,2048] 7.15 / 6.93 / 8.65, [1152,7168] 7.74 / 7.42 / 9.40, [4096,2048] 8.02 / 7.39 / 10.2,
//   but [2048,4096] 8.31 / 9.15 / 9.32;  [4608,2048] 9.61 / 10.18 / 10.82, [6144,2048] 11.18 / 10.91 / 11.89, [3072,4096] 11.43 / 13.14 / 11.40, [3584,4096] 13.78 / 13.92 /
//   12.81, [4096,4096] 15.34 / 16.18 / 14.44, [2048,7168] 13.04 / 11.76 / 11.95, [2304,7168] 14.02 / 12.76 / 13.04, [7168,2048] 13.34 / 11.61 / 13.58, but [8192,2048]
//   14.52 / 12.88 / 17.10
// More tiles than that to E2M1, whose stores of a lane's 8 codes are 4 bytes in a 128-column tile and 8 in a wider one, go with 256 columns
// and 512 threads from 1233 on (bf16, 128 / 256 columns: [10240,2048] 11.35 / 10.94, [2816,7168] 10.70 / 10.75, [5120,4096] 11.37 / 10.67, [12352,2048] 13.6 / 12.7,
// [16384,7168] 48.5 / 45.8, but [8704,2048] 9.95 / 10.30, [9216,2048] 10.30 / 10.67, [4608,4096] 10.15 / 10.42, [2560,7168] 10.22 / 10.44; fp32 [16384,7168] 86.5 / 82.6, but
// [8192,8192] 47.6 / 53.7).
// Bounds in 128 x 128 tiles:
constexpr int64_t kWideMaxTiles = 1024, kMidMaxTiles = 512, kManyMinTiles = 1233;
template <bool F32, int FMT> constexpr int64_t kWideMinTiles = FMT != TK_E2M1 ? 561 : F32 ? 833 : 641;
template <bool F32, int FMT> constexpr int64_t kMidMinTiles = F32 && FMT != TK_E2M1 ? 300 : 384;

template <typename InT, int FMT, int BM, int BK, int TW, int THREADS>
static void launch_per_block_3(const PerBlockParams &p, hipStream_t stream) {
    const dim3 grid((unsigned)((p.K + TW - 1) / TW), (unsigned)p.tiles_m), block(THREADS);
    // fp32 of at most 64 rows: each lane loads what it has, in a branch.  With few loads per lane the waits in between cost less than
    // loads of rows that do not exist and the exchange between lanes (us, without branches / this, blocks of 128 and of 32: 1 row of
    // 2560 3.05 / 2.55, 4.0 / 3.35; 40 rows 3.2 / 3.15, 4.2 / 3.75; 64 of 2816 3.3 / 3.35, 4.15 / 3.9; but 65 of 2560 3.65 / 4.4, 4.65 / 5.1).
    if constexpr (std::is_same<InT, float>::value && TW == kBlockTile) {
        if (p.M <= 64) {
            hipLaunchKernelGGL((per_block_cast_kernel<InT, FMT, BM, BK, TW, THREADS, false, true>), grid, block, 0, stream, TK_PB_LAUNCH_ARGS(p));
            return;
        }
    }
    if (p.M % kBlockTile == 0 && p.K % TW == 0)
        hipLaunchKernelGGL((per_block_cast_kernel<InT, FMT, BM, BK, TW, THREADS, true>), grid, block, 0, stream, TK_PB_LAUNCH_ARGS(p));
    else
        hipLaunchKernelGGL((per_block_cast_kernel<InT, FMT, BM, BK, TW, THREADS, false>), grid, block, 0, stream, TK_PB_LAUNCH_ARGS(p));
}

template <typename InT, int FMT, int BM, int BK>
static void launch_per_block_2(const PerBlockParams &p, hipStream_t stream) {
    const int64_t tiles = (int64_t)p.tiles_m * p.tiles_k;
    constexpr bool F32 = std::is_same<InT, float>::value;
    if (p.K % kWideTile == 0 && tiles >= kWideMinTiles<F32, FMT> && tiles <= kWideMaxTiles) {
        launch_per_block_3<InT, FMT, BM, BK, kWideTile, kWideThreads>(p, stream);
        return;
    }
    if (p.K % kMidTile == 0 && tiles >= kMidMinTiles<F32, FMT> && tiles <= kMidMaxTiles) {
        launch_per_block_3<InT, FMT, BM, BK, kMidTile, kWideThreads>(p, stream);
        return;
    }
    if constexpr (FMT == TK_E2M1 && !F32) {
        if (p.K % kMidTile == 0 && tiles >= kManyMinTiles) {
            launch_per_block_3<InT, FMT, BM, BK, kMidTile, kPerBlockThreads>(p, stream);
            return;
        }
    }
    launch_per_block_3<InT, FMT, BM, BK, kBlockTile, kPerBlockThreads>(p, stream);
}

template <typename InT, int FMT>
static hipError_t launch_per_block(const PerBlockParams &p, int bm, int bk, hipStream_t stream) {
    if (bm == 128 && bk == 128) launch_per_block_2<InT, FMT, 128, 128>(p, stream);
    else if (bm == 32 && bk == 32) launch_per_block_2<InT, FMT, 32, 32>(p, stream);
    else if (bm == 128 && bk == 32) launch_per_block_2<InT, FMT, 128, 32>(p, stream);
    else launch_per_block_2<InT, FMT, 32, 128>(p, stream);
    return hipGetLastError();
}

}  // namespace tk

using namespace tk;

extern "C" int tk_check_per_block_cast(const void *x, int x_dtype, int64_t M, int64_t K, const void *out,
                                       const void *sf, int64_t sf_ld, int fmt, int bm, int bk, int sf_layout,
                                       int round_sf, int mode) {
    if (x_dtype != TK_BF16 && x_dtype != TK_F32) return TK_ERR_BAD_DTYPE;
    if (fmt != TK_E4M3 && fmt != TK_E2M1) return TK_ERR_BAD_FORMAT;
    if (mode < TK_CAST_AND_SF || mode > TK_CAST_GIVEN_SF) return TK_ERR_BAD_MODE;
    if (sf_layout < TK_SF_ROW_F32 || sf_layout > TK_SF_COL_UE8M0) return TK_ERR_BAD_LAYOUT;
    if (mode == TK_CAST_GIVEN_SF && sf_layout != TK_SF_ROW_F32) return TK_ERR_BAD_LAYOUT;
    if (sf_layout == TK_SF_COL_UE8M0 && !round_sf) return TK_ERR_BAD_LAYOUT;
    if ((bm != 32 && bm != 128) || (bk != 32 && bk != 128)) return TK_ERR_BAD_GROUP;
    if (M < 0 || K <= 0 || K % 64 != 0) return TK_ERR_BAD_SHAPE;
    if (M > INT32_MAX - 256 || K > INT32_MAX - 256) return TK_ERR_TOO_LARGE;
    if (M == 0) return TK_OK;
    if (!x || !sf || (mode != TK_SF_ONLY && !out)) return TK_ERR_NULL_POINTER;
    if (!aligned_to(x, 16) || (mode != TK_SF_ONLY && !aligned_to(out, 8)) || !aligned_to(sf, 4)) return TK_ERR_MISALIGNED;
    const int64_t nm = (M + bm - 1) / bm, nk = (K + bk - 1) / bk;
    const int64_t need = sf_layout == TK_SF_ROW_F32 ? nk : (sf_layout == TK_SF_COL_F32 ? nm : 4 * nm);
    if (sf_ld < need) return TK_ERR_BAD_STRIDE;
    const int64_t tiles = ((M + kBlockTile - 1) / kBlockTile) * ((K + kBlockTile - 1) / kBlockTile);
    if (tiles > INT32_MAX - 8 || (M + kBlockTile - 1) / kBlockTile > 65535) return TK_ERR_TOO_LARGE;   // row tiles ride on grid.y
    return TK_OK;
}

extern "C" int tk_per_block_cast(const void *x, int x_dtype, int64_t M, int64_t K, void *out, void *sf,
                                 int64_t sf_ld, int fmt, int bm, int bk, int sf_layout, int round_sf, int mode,
                                 void *stream) {
    const int rc = tk_check_per_block_cast(x, x_dtype, M, K, out, sf, sf_ld, fmt, bm, bk, sf_layout, round_sf, mode);
    if (rc != TK_OK || M == 0) return rc;
    PerBlockParams p;
    p.x = x;
    p.out = static_cast<uint8_t *>(out);
    p.sf = SfRef{sf, sf_ld, sf_layout, (int)((M + bm - 1) / bm), (int)((K + bk - 1) / bk)};
    p.M = (int)M;
    p.K = (int)K;
    p.tiles_m = (int)((M + kBlockTile - 1) / kBlockTile);
    p.tiles_k = (int)((K + kBlockTile - 1) / kBlockTile);
    p.round_sf = round_sf;
    p.mode = mode;
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipError_t e;
    if (x_dtype == TK_BF16)
        e = fmt == TK_E4M3 ? launch_per_block<bf16_t, TK_E4M3>(p, bm, bk, s) : launch_per_block<bf16_t, TK_E2M1>(p, bm, bk, s);
    else
        e = fmt == TK_E4M3 ? launch_per_block<float, TK_E4M3>(p, bm, bk, s) : launch_per_block<float, TK_E2M1>(p, bm, bk, s);
    return (int)e;
}
