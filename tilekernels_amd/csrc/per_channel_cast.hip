// Per-channel (N tokens x 1 column, N in {32, 128}) E4M3 cast for gfx950, with the fusions the
// reference offers around it: row gather (pos_to_token), dequantisation of an E4M3 input with 1 x 128
// scales, SwiGLU in front, and a transposed ([K, M]) output.
//
// A workgroup of 8 waves owns a 128-token x 256-column tile (of 4 waves a 128 x 128 tile where the wide tiles are too few
// for the GPU) and keeps it in registers between the amax and the conversion, so HBM is read once.  A run of LANES = 32 (16)
// lanes x 8 columns = 256 (128) columns takes 8 consecutive tokens: run i of the workgroup holds tokens 8 i + p, p = 0..7.
// A lane therefore owns 8 columns over 8 tokens and reduces |x| down its columns without any cross-lane
// step; the 16 partial maxima per column (one per run) meet in LDS, one thread per column derives
// the scale(s) of column c (one division per scale in the whole workgroup, stored as one coalesced
// run) and hands the multipliers back through LDS.
//   plain output      : a lane converts 8 columns of a token -> one 8-byte store, 256 (128) bytes per run
//   transposed output : a lane converts 8 tokens of a column -> 8 bytes of an output row; the tile is
//                       turned in LDS ([columns][128 tokens] bytes) and leaves as 128-byte row pieces
//
// Reference semantics: tile_kernels/quant/per_channel_cast_fused_kernel.py:16-203,
// per_channel_cast_and_transpose_kernel.py:8-123,
// swiglu_forward_and_per_channel_cast_and_transpose_kernel.py:9-231; oracle
// tile_kernels/torch/per_channel_cast_fused.py and tile_kernels/torch/cast.py with block (N, 1).
#include "swiglu_math.hpp"
#include "tk_device.hpp"
#include "tk_host.hpp"

namespace tk {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kPcTileM = 128;
// Consecutive tokens per lane.  With 4 (1024 threads per tile) every mode measured slower on MI355X at
// [8192, 4096]: plain 17.7 -> 18.3 us, FP8 input 13.4 -> 14.6, transposed 21.1 -> 24.0, SwiGLU 17.3 -> 18.0.
constexpr int kPcRows = 8;
constexpr int kPcParts = kPcTileM / kPcRows;             // runs of lanes per tile = partial maxima per column: 16
// Turned tile in LDS: one row of 128 token bytes per column, rows 144 bytes apart.  A lane writes the 8
// tokens it holds of column 8 hl + j as one 8-byte word; left at its natural place (8 part) the 32
// lanes of a half-wave would meet in two (LANES = 16: four) of the 32 8-byte bank pairs (rows 8 x 144 bytes apart).  So
// the 16-byte unit of a row is rotated by (hl >> 1) & 7 and the two halves of the unit are exchanged
// when hl >= 16: with the row pitch supplying hl & 1, the five bits of hl (LANES = 16: its four bits and the parity of the run,
// which chooses the half of the unit) land in five different bits of the bank-pair index and a half-wave's writes touch every
// bank pair once.  Units stay whole, so
// the reader still takes 16 bytes at a time.
constexpr int kPcPitch = kPcTileM + 16;

enum { PC_BF16 = 0, PC_E4M3 = 1, PC_SWIGLU = 2, PC_F32 = 3 };

struct PerChannelParams {
    const void *x;
    const float *x_sf;
    const int32_t *pos_to_token;
    uint8_t *out;
    float *out_sf;
    int num_tokens, K, M;      // input rows, columns (of the output), output rows
    int tiles_k;
    int round_sf, use_clamp;
    float clamp;
};

#define TK_PC_KERNEL_ARGS                                                                                          \
    const void *a_x, uint8_t *a_out, float *a_out_sf, const float *a_x_sf, const int32_t *a_p2t, int a_T, int a_K, \
        int a_M, int a_tiles_k, int a_round_sf, int a_use_clamp, float a_clamp
#define TK_PC_KERNEL_UNPACK \
    const PerChannelParams p{a_x, a_x_sf, a_p2t, a_out, a_out_sf, a_T, a_K, a_M, a_tiles_k, a_round_sf, a_use_clamp, a_clamp}
#define TK_PC_LAUNCH_ARGS(p) \
    (p).x, (p).out, (p).out_sf, (p).x_sf, (p).pos_to_token, (p).num_tokens, (p).K, (p).M, (p).tiles_k, (p).round_sf, (p).use_clamp, (p).clamp

// What bounds the SwiGLU form is half memory, half arithmetic: 1077 vector instructions per lane (64 elements), 128 of them exponentials and
// reciprocals.  They were 1402 while the clamp was compiled in for every call (at infinity where there was none), the rounded
// activations were unpacked again for their maxima, registers were cleared for lanes beyond the matrix, and every row's address was a
// product.  us on MI355X, before / after, SwiGLU and bf16 operand together: [768, 2 x 3456] and [768, 3328] 9.3 / 8.65, [2560, 2 x 2560] and
// [2560, 4096] 16.1 / 15.1, [8064, 2 x 2048] and [8064, 4096] 35.0 / 34.3.  (With fewer workgroups resident, so that one's stores meet
// another's loads: 39 to 42.)
template <int MODE> struct PcRaw { typedef Raw8<bf16_t> type; };
template <> struct PcRaw<PC_E4M3> { typedef Raw8<e4m3in_t> type; };
template <> struct PcRaw<PC_F32> { typedef Raw8<float> type; };

// Makes the compiler treat the packed input as redefined here, so that what was unpacked from it before
// cannot be kept alive across this point.
__device__ __forceinline__ void forget_unpacked(Raw8<bf16_t> &r) { asm volatile("" : "+v"(r.w)); }
__device__ __forceinline__ void forget_unpacked(Raw8<e4m3in_t> &r) { asm volatile("" : "+v"(r.w)); }
__device__ __forceinline__ void forget_unpacked(Raw8<float> &) {}   // nothing is unpacked: the registers are the values

__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
}

// CLAMP: of the SwiGLU's inputs.
template <int MODE, int NPT, bool TRANS, bool GATHER, int LANES, bool CLAMP = false>
__global__ __launch_bounds__(LANES * kPcParts, 4) void per_channel_cast_kernel(TK_PC_KERNEL_ARGS) {
    TK_PC_KERNEL_UNPACK;
    constexpr int kPcTileK = LANES * 8, kPcThreads = LANES * kPcParts;
    constexpr int NB = kPcTileM / NPT;          // scale blocks per tile along the tokens: 1 or 4
    typedef typename PcRaw<MODE>::type Raw;
    // the partial maxima are dead once the scales exist (second barrier), so the turned tile reuses their space
    constexpr int kPartBytes = kPcParts * kPcTileK * 4, kTurnedBytes = TRANS ? kPcTileK * kPcPitch : 0;
    __shared__ __attribute__((aligned(16))) uint8_t lds[kPartBytes > kTurnedBytes ? kPartBytes : kTurnedBytes];
    __shared__ __attribute__((aligned(16))) float inv_s[NB][kPcTileK];
    float (*part)[kPcTileK] = reinterpret_cast<float (*)[kPcTileK]>(lds);    // [run][column]
    uint8_t *turned = lds;

    // 2-D grid (x = column tile, y = token tile); the FP8-input mode runs on a 1-D grid that it reorders
    int tile_m = blockIdx.y, tile_k = blockIdx.x;
    if constexpr (MODE == PC_E4M3) {
        tile_m = blockIdx.x / p.tiles_k;
        tile_k = blockIdx.x - tile_m * p.tiles_k;
        // Workgroups are dealt to the 8 XCDs (each with its own L2) round-robin.  The tiles of one token
        // range share the 128-byte lines of the input scales, so they are given to one XCD: 8 token
        // ranges advance side by side, one per XCD.  (Without this the scale lines are fetched 8 times.)
        const int tiles_m = (p.M + kPcTileM - 1) / kPcTileM, striped = (tiles_m / 8) * 8 * p.tiles_k;
        if ((int)blockIdx.x < striped) {
            const int q = blockIdx.x >> 3;
            tile_k = q % p.tiles_k;
            tile_m = (q / p.tiles_k) * 8 + (blockIdx.x & 7);
        }
    }
    const int lane = threadIdx.x & 63, run = wave_id() * (64 / LANES) + lane / LANES, hl = lane % LANES;
    const int col0 = tile_k * kPcTileK, col = col0 + hl * 8;
    const bool col_ok = col < p.K;
    const int tok0 = tile_m * kPcTileM + run * kPcRows;
    const bool rows_ok = tok0 < p.M;            // M is a multiple of 16: all 8 tokens of a lane or none
    const int64_t in_ld = MODE == PC_SWIGLU ? 2 * (int64_t)p.K : p.K;

    // ---- load (and, for SwiGLU, activate) 8 tokens x 8 columns.  No lane branches around its loads: one beyond the last token reads
    // the last 8 tokens, whose scale block is its own or one that is not stored, one beyond the last column the last 8 columns.  (M is a
    // multiple of 16, K of 8.)  A gathered row with a negative index is read from row 0 and zeroed by value.
    const int tok_in = min(tok0, p.M - kPcRows), col_in = min(col, p.K - 8);
    Raw raw[kPcRows];
    float m[8];          // |x| maxima down this lane's 8 columns
#pragma unroll
    for (int j = 0; j < 8; ++j) m[j] = 0.0f;
    if constexpr (MODE == PC_SWIGLU) {
        // all sixteen loads of the lane go out before the first activation is evaluated (issuing them in batches of
        // 4 or 2 tokens brings the kernel from 92 to 67 / 61 VGPRs and more waves per SIMD, but measured 18-19 us
        // against 16.8 us for bf16 [8192, 4096])
        Raw8<bf16_t> rg[kPcRows], ru[kPcRows];
        const uint16_t *xr = reinterpret_cast<const uint16_t *>(p.x) + tok_in * in_ld + col_in;
#pragma unroll
        for (int r = 0; r < kPcRows; ++r, xr += in_ld) {
            rg[r].load(xr);
            vmem_issue_gap();
            ru[r].load(xr + p.K);
            vmem_issue_gap();
        }
        __builtin_amdgcn_sched_barrier(0);
        float cl = 0.0f, lo = 0.0f;
        if constexpr (CLAMP) {
            // the clamp lies beyond the preloaded arguments: touched only now, behind the loads
            cl = p.clamp;
            asm volatile("" : "+s"(cl));
            lo = cl >= 0.0f ? -cl : cl;      // (a negative limit makes every element the limit, as the two-step form does)
        }
#pragma unroll
        for (int r = 0; r < kPcRows; ++r) {
            float g[8], u[8], a[8];
            rg[r].get(g);
            ru[r].get(u);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if constexpr (CLAMP) {
                    g[i] = __builtin_fminf(g[i], cl);
                    u[i] = __builtin_amdgcn_fmed3f(u[i], lo, cl);      // min(max(u, -cl), cl) in one instruction
                }
                a[i] = silu_mul<bf16_t>(g[i], u[i]);
                m[i] = __builtin_fmaxf(m[i], __builtin_fabsf(a[i]));
            }
            // the activation is rounded to bf16 before it is quantised, as in the reference
            raw[r].w = u32x4{pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]), pack_bf16x2(a[4], a[5]), pack_bf16x2(a[6], a[7])};
        }
        // the largest rounded magnitude is the rounded largest one
        Raw8<bf16_t> rounded;
        rounded.w = u32x4{pack_bf16x2(m[0], m[1]), pack_bf16x2(m[2], m[3]), pack_bf16x2(m[4], m[5]), pack_bf16x2(m[6], m[7])};
        rounded.get(m);
    } else {
        // (the gather indices of all rows are asked for before the first row's data: a load whose address hangs on a loaded value
        // waits for every load issued before it)
        int gathered[kPcRows];
        bool valid[kPcRows];
        if constexpr (GATHER) {
#pragma unroll
            for (int r = 0; r < kPcRows; ++r) gathered[r] = p.pos_to_token[tok_in + r];
        }
#pragma unroll
        for (int r = 0; r < kPcRows; ++r) {
            int src = tok_in + r;
            valid[r] = true;
            if constexpr (GATHER) {
                src = gathered[r];
                valid[r] = src >= 0 && src < p.num_tokens;
                src = valid[r] ? src : 0;
            }
            if constexpr (MODE == PC_E4M3) {
                raw[r].load(reinterpret_cast<const uint8_t *>(p.x) + (int64_t)src * in_ld + col_in);
                vmem_issue_gap();
                raw[r].s = p.x_sf[(int64_t)src * (p.K >> 7) + (col_in >> 7)];
                vmem_issue_gap();
            } else if constexpr (MODE == PC_F32) {
                raw[r].load(reinterpret_cast<const float *>(p.x) + (int64_t)src * in_ld + col_in);
                vmem_issue_gap();
            } else {
                raw[r].load(reinterpret_cast<const uint16_t *>(p.x) + (int64_t)src * in_ld + col_in);
                vmem_issue_gap();
            }
        }
        // (rows without a source are cleared once all loads are out: clearing a register a load is still to fill means waiting for it)
        if constexpr (GATHER) {
#pragma unroll
            for (int r = 0; r < kPcRows; ++r)
                if (!valid[r]) raw[r].zero();
        }
#pragma unroll
        for (int r = 0; r < kPcRows; ++r) {
            float v[8];
            raw[r].get(v);
#pragma unroll
            for (int j = 0; j < 8; ++j) m[j] = __builtin_fmaxf(m[j], __builtin_fabsf(v[j]));
        }
        // the tile is unpacked a second time after the scales are known; without this the compiler keeps
        // all 64 unpacked values alive across the two barriers instead
#pragma unroll
        for (int r = 0; r < kPcRows; ++r) forget_unpacked(raw[r]);
    }
    {
        u32x4 *dst = reinterpret_cast<u32x4 *>(&part[run][hl * 8]);
        dst[0] = u32x4{f2u(m[0]), f2u(m[1]), f2u(m[2]), f2u(m[3])};
        dst[1] = u32x4{f2u(m[4]), f2u(m[5]), f2u(m[6]), f2u(m[7])};
    }
    __syncthreads();

    // ---- thread c: scale(s) of column c
    if (threadIdx.x < kPcTileK) {
        const int c = threadIdx.x;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            float a = 0.0f;
#pragma unroll
            for (int i = 0; i < kPcParts / NB; ++i) a = __builtin_fmaxf(a, part[b * (kPcParts / NB) + i][c]);
            const Scale sc = make_scale<448>(a, Fmt<TK_E4M3>::floor_, p.round_sf != 0);
            inv_s[b][c] = sc.inv;
            const int tok = tile_m * kPcTileM + b * NPT;
            if (tok < p.M && col0 + c < p.K) st_stream4(p.out_sf + (int64_t)(tok / NPT) * p.K + col0 + c, f2u(sc.sf));
        }
    }
    __syncthreads();

    float inv[8];
    {
        const u32x4 *src = reinterpret_cast<const u32x4 *>(&inv_s[NB == 1 ? 0 : (run * kPcRows) / 32][hl * 8]);
        const u32x4 a = src[0], b = src[1];
        inv[0] = u2f(a.x); inv[1] = u2f(a.y); inv[2] = u2f(a.z); inv[3] = u2f(a.w);
        inv[4] = u2f(b.x); inv[5] = u2f(b.y); inv[6] = u2f(b.z); inv[7] = u2f(b.w);
    }

    if constexpr (!TRANS) {
#pragma unroll
        for (int r = 0; r < kPcRows; ++r) {
            float v[8], q[8];
            raw[r].get(v);
#pragma unroll
            for (int j = 0; j < 8; ++j) q[j] = v[j] * inv[j];
            if (rows_ok && col_ok) st_stream8(p.out + (int64_t)(tok0 + r) * p.K + col, pack_e4m3x8<false>(q));
        }
    } else {
        // codes of the lane's 8 consecutive tokens per column: token pairs fill the 16-bit halves of a dword
        uint32_t acc[8][2];
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            float v0[8], v1[8], v2[8], v3[8];
            raw[4 * d].get(v0);
            raw[4 * d + 1].get(v1);
            raw[4 * d + 2].get(v2);
            raw[4 * d + 3].get(v3);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float a = v0[j] * inv[j], b = v1[j] * inv[j];
                const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, (int)f2u(a), false);      // (any register serves as the half that the next one fills)
                acc[j][d] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(v2[j] * inv[j], v3[j] * inv[j], lo, true);
            }
        }
        {
            const int unit = ((run >> 1) + (hl >> 1)) & 7, low = (run & 1) ^ (hl >> 4);
            uint8_t *dst = &turned[hl * 8 * kPcPitch + unit * 16 + low * 8];
#pragma unroll
            for (int j = 0; j < 8; ++j) *reinterpret_cast<u32x2 *>(dst + j * kPcPitch) = u32x2{acc[j][0], acc[j][1]};
        }
        __syncthreads();
        // 8 lanes x 16 bytes = the 128 tokens of one output row; a wave stores 8 rows per step
        const int chunk = threadIdx.x & 7;
        const int tok = tile_m * kPcTileM + chunk * 16;
        // Behind the SwiGLU a launch of more tiles than fit the GPU at a time (two to a CU) writes through: 128-byte pieces of its output rows
        // that stay behind in the L2 leave it in no order.  us, non-temporal / write-through, three sets of inputs in rotation (twelve):
        // [8192, 2 x 8320] 65.2 / 58.8 (66.0 / 66.8), [16384, 2 x 2048] 31.6 / 30.4 (32.2 / 30.7), [12288, 2 x 2560] 29.5 / 28.0 (30.0 / 28.1), [4480,
        // 2 x 6144] 26.4 / 25.8 (26.7 / 25.9); in one round [8064, 2 x 2048] 16.4 / 16.2 (16.5 / 18.1).  (Neighbouring token tiles side by side in
        // the grid, 2, 4 or 8, on neighbouring XCDs or on one, so that pieces of one row meet: 1 to 5 % slower.)
        const bool through = MODE == PC_SWIGLU && LANES == 32 && p.tiles_k * ((p.M + kPcTileM - 1) / kPcTileM) > 512;
#pragma unroll
        for (int i = 0; i < kPcTileK / (kPcThreads / 8); ++i) {
            const int h = (threadIdx.x >> 3) + (kPcThreads / 8) * i;
            if (col0 + h < p.K && tok < p.M) {
                const int unit = (chunk + (h >> 4)) & 7;
                u32x4 d = *reinterpret_cast<const u32x4 *>(&turned[h * kPcPitch + unit * 16]);
                if (LANES == 32 && i >= 2) d = u32x4{d.z, d.w, d.x, d.y};          // rows of the lanes hl >= 16: h >= 128
                // (write-through stores against non-temporal ones, bf16 [8192, 4096] on MI355X: plain and FP8 input 19.6 -> 19.2 us, ordinary
                // stores 19.6 and 18.4 us; behind the SwiGLU see `through`)
                if (MODE != PC_SWIGLU || through) st_stream16(p.out + (int64_t)(col0 + h) * p.M + tok, d);
                else __builtin_nontemporal_store(d, reinterpret_cast<u32x4 *>(p.out + (int64_t)(col0 + h) * p.M + tok));
            }
        }
    }
}

// Gathered E4M3 rows: whether a launch whose output is mostly padding or tokens that other rows repeat takes narrow tiles.  Up to 16383 tokens,
// where narrow tiles can go in column order (below): from 9100 tokens [13120, 2560] wide / narrow 12.5 / 11.4 us, cold 14.3 / 15.2.  Beyond that
// they would not, and wide tiles with ordinary loads serve repeated rows better; us, narrow / wide (wide with non-temporal loads), three sets of inputs in
// rotation | twelve:  16384 tokens twice each, K = 2048 23.6 / 23.9 (28.5) | 29.8 / 27.4 (29.0), K = 7168 90.0 / 83.1 (88.5) | 91.5 / 84.9 (88.7);  eight times
// each, K = 2048 72.4 / 71.7 (91.9) | 80.6 / 77.4 (91.5), K = 7168 295 / 286 (323) | 295 / 287 (324);  32768 twice, K = 2048 42.3 / 43.0 (51.1) | 52.8 / 49.6 (51.0),
// K = 7168 179 / 167 (170) | 179 / 167 (171);  20000 once each among 65536 rows, K = 2048 29.3 / 30.0 (33.5) | 36.3 / 34.9 (34.2)
__host__ __device__ inline bool gather_repeats(int num_tokens, int M) { return num_tokens < 16384 && 4 * (int64_t)M >= 7 * (int64_t)num_tokens; }
// and whether those tiles go in column order, each XCD down a column of its own: a column tile of all tokens (256 bytes of each, so up to 16383 of
// them) stays in the XCD's 4 MB L2 until the next expert's rows ask for it.  us, striped / in column order, three sets | twelve:  5401 tokens -> [10112,
// 7168] 21.6 / 19.2, 8192 -> [18432, 7168] 37.1 / 33.0, 14336 six times each, K = 2048 54.4 / 41.9 | 59.1 / 54.8;  narrow rows, 6000 twice, K = 512 4.7 / 4.4 | 5.4 /
// 5.3, 8192 twice 5.8 / 5.9 | 6.6 / 6.8.  Fewer tokens than 4096 gain by it where they are repeated (3000 twice, K = 7168 16.0 / 13.6 | 19.7 / 19.3; 1024 twice 8.5 /
// 7.7 | 8.5 / 8.2) and lose where they stand between padding, which for so few tokens of several experts is the rule, whatever their bytes (88 -> [31616, 7168]
// 40.4 / 47.4, 1202 -> [18048, 6144] 22.2 / 24.9 | 22.4 / 25.6, 3000 -> [32768, 7168], 21 MB of rows, 42.8 / 47.3 | 44.1 / 51.0; 6000 -> [32768, 4096] 27.1 / 26.9 | 29.7 / 30.3).
__host__ __device__ inline bool gather_by_columns(int num_tokens, int M) { return gather_repeats(num_tokens, M) && num_tokens >= 4096; }

// Offset beyond the end of any buffer, also with a lane's part of up to 496 bytes added to it.
constexpr uint32_t kPcNowhere = 0xFFFFFC00u;

// out[r] = v of lane 8 g + r, in every lane of lanes 8 g .. 8 g + 7
__device__ __forceinline__ void deal_rows(uint32_t (&out)[kPcRows], uint32_t v) {
#define TK_PC_DEAL(r) out[r] = (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, (r) << 5 | 0x18)
    TK_PC_DEAL(0); TK_PC_DEAL(1); TK_PC_DEAL(2); TK_PC_DEAL(3);
    TK_PC_DEAL(4); TK_PC_DEAL(5); TK_PC_DEAL(6); TK_PC_DEAL(7);
#undef TK_PC_DEAL
}

// Write-through store of 16 codes.  (The conversion that makes a code fills half a register, and what reads it next has to stay one wait
// state away; the compiler keeps that distance from instructions it knows, this one keeps it by itself.)
__device__ __forceinline__ void st_codes16(void *p, u32x4 v) {
    asm volatile("s_nop 0" : "+v"(v));
    st_stream16(p, v);
}

// E4M3 input with 1 x 128 scales, plain (not transposed) output, with 16 codes per lane instead of 8: a workgroup of 512
// threads owns 128 tokens x 512 columns, half a wave (32 lanes x 16 columns) takes 8 consecutive tokens, and every
// load and store instruction of a lane moves 16 bytes (8 bytes per lane make a half-wave's instruction 256 bytes
// long; measured on MI355X at [8192, 4096]: 13.8 us that way, 12.8 us this way).  The rest is the kernel above: maxima down the lane's columns, the 16 partial maxima per column meet in LDS,
// thread c derives the scale(s) of column c and hands the multipliers back.
// LANES = 16: 256 threads, 128 x 256 tiles, where the wide tiles are too few for the GPU and for gathers with much reuse or padding.
//
// Gathered rows.  What bounds a gather is its reads of rows that other tiles read too: every token is fetched once per expert it went to,
// and non-temporal loads fetch it from HBM each time; with ordinary loads the second read is served by a cache.  Padding rows read nothing:
// the input is a buffer in scalar registers, their offset lies beyond its end, and what is read there is zero (reads of some row in their
// place all went to the same lines).  A half-wave's scales and source rows come with one load each, lane (group, row) holding row `row`'s,
// and are dealt out within the half-wave.  us on MI355X, all rows by non-temporal loads, padding from row 0 / this, three sets of inputs in
// rotation (twelve, which no cache holds):
//   experts' rows of 7168 from 5401 tokens, [10112] 29.1 / 19.2 (29.8 / 28.5);  two copies each of 8192 tokens, [18432] 49.5 / 33.0 (49.7 / 47.7)
//   mostly padding: 244 tokens -> [32768, 3968] 40.9 / 25.8 (43.0 / 25.7), 1202 -> [18048, 6144] 41.0 / 23.9 (40.2 / 24.0), 928 -> [32768, 3712]
//   42.6 / 24.4 (43.6 / 24.0);  little of either: 16600 -> [17408, 6144] 42.6 / 42.6 (43.0 / 44.4), 19800 -> [28800, 4096] 43.8 / 42.4 (44.1 / 43.3)
// So rows that are about as many as the tokens, each read about once, keep the non-temporal loads.
// SRC: where rows come from.  PC_IN_ORDER: those of the output; PC_GATHERED; PC_GATHERED_ONCE: with non-temporal loads; PC_GATHERED_FAR:
// from more than a buffer's 4 GB, by addresses.
// THROUGH: write-through stores.  Where the output is short, nothing is left to be written back when the launch ends ([4096, 4096] 6.2 / 5.4
// us, [16384, 1024] 6.1 / 5.4, but [8128, 2560] from cold inputs 8.7 / 10.9, [10112, 7168] 21.6 / 30.5).
enum { PC_IN_ORDER = 0, PC_GATHERED = 1, PC_GATHERED_ONCE = 2, PC_GATHERED_FAR = 3 };
template <int NPT, int SRC, int LANES, bool THROUGH>
__global__ __launch_bounds__(LANES * kPcParts, 4) void per_channel_cast_fp8in_kernel(TK_PC_KERNEL_ARGS) {
    TK_PC_KERNEL_UNPACK;
    constexpr bool GATHER = SRC != PC_IN_ORDER, BUFFER = SRC == PC_GATHERED || SRC == PC_GATHERED_ONCE;
    constexpr int kPcWideK = LANES * 16;
    constexpr int NB = kPcTileM / NPT;
    __shared__ __attribute__((aligned(16))) float part[kPcParts][kPcWideK];
    __shared__ __attribute__((aligned(16))) float inv_s[NB][kPcWideK];

    // the tiles of one token range share the 128-byte lines of the input scales: 8 token ranges advance side by
    // side, one per XCD (workgroups are dealt to the XCDs round-robin)
    const int tiles_m = (p.M + kPcTileM - 1) / kPcTileM;
    int tile_m = blockIdx.x / p.tiles_k, tile_k = blockIdx.x - tile_m * p.tiles_k;
    if (SRC == PC_GATHERED && LANES == 16 && gather_by_columns(p.num_tokens, p.M)) {
        // the tiles in column order, cut into one consecutive eighth per XCD
        const int tiles = (int)gridDim.x, xcd = blockIdx.x & 7;
        const int at = xcd * (tiles >> 3) + min(xcd, tiles & 7) + (int)(blockIdx.x >> 3);
        tile_k = at / tiles_m;
        tile_m = at - tile_k * tiles_m;
    } else if (const int striped = (tiles_m / 8) * 8 * p.tiles_k; (int)blockIdx.x < striped) {
        const int q = blockIdx.x >> 3;
        tile_k = q % p.tiles_k;
        tile_m = (q / p.tiles_k) * 8 + (blockIdx.x & 7);
    }
    const int lane = threadIdx.x & 63, run = wave_id() * (64 / LANES) + lane / LANES, hl = lane % LANES;
    const int col0 = tile_k * kPcWideK, col = col0 + hl * 16;
    const bool col_ok = col < p.K;              // K is a multiple of 128: all 16 columns of a lane or none
    const int tok0 = tile_m * kPcTileM + run * kPcRows;
    const bool rows_ok = tok0 < p.M;            // M is a multiple of 16: all 8 tokens of a lane or none

    Raw8<e4m3in_t> lo[kPcRows], hi[kPcRows];
    if constexpr (BUFFER) {
        constexpr int kHint = SRC == PC_GATHERED_ONCE ? 2 : 0;      // 2: non-temporal
        const uint32_t row_bytes = (uint32_t)p.K, sf_bytes = (uint32_t)(p.K >> 7) * 4u;
        const __amdgpu_buffer_rsrc_t x = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(reinterpret_cast<const uint8_t *>(p.x)) + col0, 0,
                                                                           (int)((uint32_t)p.num_tokens * row_bytes - (uint32_t)col0), 0x00020000);
        const __amdgpu_buffer_rsrc_t x_sf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.x_sf), 0, (int)((uint32_t)p.num_tokens * sf_bytes), 0x00020000);
        // lane (g, r) of the run: row r, and the scale of its columns 128 g ..; whether there are such columns is the same for its 8 lanes
        const int src = p.pos_to_token[rows_ok ? tok0 + (hl & 7) : 0];
        const bool live = rows_ok && col_ok && src >= 0 && src < p.num_tokens;
        uint32_t offs[kPcRows];
        deal_rows(offs, live ? (uint32_t)src * row_bytes : kPcNowhere);
        u32x4 w[kPcRows];
#pragma unroll
        for (int r = 0; r < kPcRows; ++r) {
            w[r] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(x, offs[r] + (uint32_t)(hl * 16), 0, kHint));
            vmem_issue_gap();
        }
        const uint32_t s = __builtin_amdgcn_raw_buffer_load_b32(x_sf, live ? (uint32_t)src * sf_bytes + (uint32_t)(col >> 7) * 4u : kPcNowhere, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        uint32_t scales[kPcRows];
        deal_rows(scales, s);
#pragma unroll
        for (int r = 0; r < kPcRows; ++r) {
            lo[r].w = u32x2{w[r].x, w[r].y};
            hi[r].w = u32x2{w[r].z, w[r].w};
            lo[r].s = hi[r].s = u2f(scales[r]);
        }
    } else {
#pragma unroll
        for (int r = 0; r < kPcRows; ++r) { lo[r].zero(); hi[r].zero(); }
        if (rows_ok && col_ok) {
            // (gather indices of all rows first: see per_channel_cast_kernel)
            int gathered[kPcRows];
            if constexpr (GATHER) {
#pragma unroll
                for (int r = 0; r < kPcRows; ++r) gathered[r] = p.pos_to_token[tok0 + r];
            }
#pragma unroll
            for (int r = 0; r < kPcRows; ++r) {
                int src = tok0 + r;
                bool valid = true;
                if constexpr (GATHER) {
                    src = gathered[r];
                    valid = src >= 0 && src < p.num_tokens;
                    src = valid ? src : 0;
                }
                const u32x4 w = ld_stream16(reinterpret_cast<const uint8_t *>(p.x) + (int64_t)src * p.K + col);
                vmem_issue_gap();
                lo[r].w = u32x2{w.x, w.y};
                hi[r].w = u32x2{w.z, w.w};
                lo[r].s = hi[r].s = p.x_sf[(int64_t)src * (p.K >> 7) + (col >> 7)];
                vmem_issue_gap();
                gathered[r] = valid ? 1 : 0;
            }
            if constexpr (GATHER) {      // (cleared once all loads are out)
#pragma unroll
                for (int r = 0; r < kPcRows; ++r)
                    if (!gathered[r]) { lo[r].zero(); hi[r].zero(); }
            }
        }
    }

    float m[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) m[j] = 0.0f;
#pragma unroll
    for (int r = 0; r < kPcRows; ++r) {
        float a[8], b[8];
        lo[r].get(a);
        hi[r].get(b);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            m[j] = __builtin_fmaxf(m[j], __builtin_fabsf(a[j]));
            m[8 + j] = __builtin_fmaxf(m[8 + j], __builtin_fabsf(b[j]));
        }
    }
    // the tile is decoded a second time after the scales are known, instead of 128 values kept alive across the barriers
#pragma unroll
    for (int r = 0; r < kPcRows; ++r) { forget_unpacked(lo[r]); forget_unpacked(hi[r]); }
    {
        u32x4 *dst = reinterpret_cast<u32x4 *>(&part[run][hl * 16]);
#pragma unroll
        for (int q = 0; q < 4; ++q) dst[q] = u32x4{f2u(m[4 * q]), f2u(m[4 * q + 1]), f2u(m[4 * q + 2]), f2u(m[4 * q + 3])};
    }
    __syncthreads();

    {
        const int c = threadIdx.x;               // as many threads as columns
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            float a = 0.0f;
#pragma unroll
            for (int i = 0; i < kPcParts / NB; ++i) a = __builtin_fmaxf(a, part[b * (kPcParts / NB) + i][c]);
            const Scale sc = make_scale<448>(a, Fmt<TK_E4M3>::floor_, p.round_sf != 0);
            inv_s[b][c] = sc.inv;
            const int tok = tile_m * kPcTileM + b * NPT;
            if (tok < p.M && col0 + c < p.K) st_stream4(p.out_sf + (int64_t)(tok / NPT) * p.K + col0 + c, f2u(sc.sf));
        }
    }
    __syncthreads();

    float inv[16];
    {
        const u32x4 *src = reinterpret_cast<const u32x4 *>(&inv_s[NB == 1 ? 0 : (run * kPcRows) / 32][hl * 16]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const u32x4 v = src[q];
            inv[4 * q] = u2f(v.x); inv[4 * q + 1] = u2f(v.y); inv[4 * q + 2] = u2f(v.z); inv[4 * q + 3] = u2f(v.w);
        }
    }
#pragma unroll
    for (int r = 0; r < kPcRows; ++r) {
        float a[8], b[8];
        lo[r].get(a);
        hi[r].get(b);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            a[j] = a[j] * inv[j];
            b[j] = b[j] * inv[8 + j];
        }
        const u32x2 x0 = pack_e4m3x8<false>(a), x1 = pack_e4m3x8<false>(b);
        if (rows_ok && col_ok) {
            uint8_t *dst = p.out + (int64_t)(tok0 + r) * p.K + col;
            if constexpr (THROUGH) st_codes16(dst, u32x4{x0.x, x0.y, x1.x, x1.y});
            else __builtin_nontemporal_store(u32x4{x0.x, x0.y, x1.x, x1.y}, reinterpret_cast<u32x4 *>(dst));
        }
    }
}

// Wide tiles from which on a launch takes them; with fewer it takes narrow ones (16 lanes per run, twice as many workgroups of half the
// size).  An MI355X has 256 compute units.  What computes more per byte (the SwiGLU, E4M3 input, the turn of a transposed output,
// gathered bf16 rows) is better off in narrow tiles as long as wide ones leave compute units without work; where loads and stores are
// all there is, narrow tiles lose already where some units hold two of them and others one, fp32 (a wide tile is 128 KB) as soon as any
// unit does.  Measured on MI355X, us per call, wide / narrow:
//   SwiGLU transposed [128, 4096] 7.4 / 5.1, [1024, 2048] (64 wide tiles) 7.9 / 5.6, [4096, 1408] (192) 8.8 / 8.5, [896, 8192] (224) 9.15 / 9.1,
//   [16256, 1024] (508) 16.6 / 16.4, [12800, 3072] (1200) 37.4 / 39.9; bf16 transposed [1024, 7168] (224) 5.3 / 4.85, [2304, 2560] (180)
//   5.05 / 4.45, [16256, 1024] (508) 9.2 / 9.65; E4M3 input [4608, 1408] (108) 6.2 / 5.1, [2048, 7168] (224) 6.7 / 6.6, [4096, 4096] (256)
//   7.25 / 7.6, [13120, 2560] (515) 13.8 / 15.0; bf16 gathered [2048, 3072] (192) 4.3 / 3.9, [1152, 7168] (252) 4.6 / 4.2;
//   bf16 [2048, 2048] (128) 3.5 / 2.95, [4096, 1280] (160) 4.2 / 4.1, [3072, 1792] (168) 4.2 / 4.05, [1024, 5632] (176) 4.34 / 4.41,
//   [4096, 1536] (192) 4.4 / 4.7, [2048, 3584] (224) 4.6 / 5.3; fp32, gathered or not, [2048, 2048] (128) 7.0 / 5.3, [512, 8448] (132) 7.4 / 7.9,
//   [1024, 5120] (160) 7.2 / 8.1, [2048, 3584] (224) 8.0 / 9.2.
// (Runs of 8 lanes: [128, 4096] 4.9, [1024, 7168] 5.7; 4 tokens per lane instead of 8, E4M3 input: [10112, 7168] 29.0 / 32.0.)
template <int MODE> static int64_t wide_tiles_from(bool transpose, bool gather) {
    if (MODE == PC_F32) return 129;
    return MODE != PC_BF16 || transpose || gather ? 256 : 176;
}

constexpr int64_t kPcThrough = 16 << 20;      // bytes of output up to which gathered codes are written through
// More input than a buffer can hold, and rows that are read about once (see the kernel).
static bool gather_far(const PerChannelParams &p) { return (int64_t)p.num_tokens * p.K > (int64_t)kPcNowhere; }
static bool gather_once(const PerChannelParams &p) { return 4 * (int64_t)p.M < 5 * (int64_t)p.num_tokens; }

template <int MODE, int NPT, int LANES>
static void launch_per_channel_3(const PerChannelParams &a, bool transpose, hipStream_t stream) {
    PerChannelParams p = a;
    const int tiles_m = (p.M + kPcTileM - 1) / kPcTileM;
    const dim3 block(LANES * kPcParts);
    if constexpr (MODE == PC_E4M3) {
        if (!transpose && aligned_to(p.x, 16) && aligned_to(p.out, 16)) {
            p.tiles_k = (p.K + LANES * 16 - 1) / (LANES * 16);
            const dim3 grid((unsigned)(tiles_m * p.tiles_k));
#define TK_PC_FP8_LAUNCH(SRC, T) \
    hipLaunchKernelGGL((per_channel_cast_fp8in_kernel<NPT, SRC, LANES, T>), grid, block, 0, stream, TK_PC_LAUNCH_ARGS(p))
            if (!p.pos_to_token) TK_PC_FP8_LAUNCH(PC_IN_ORDER, false);
            else if (LANES == 32 && gather_far(p)) TK_PC_FP8_LAUNCH(LANES == 32 ? PC_GATHERED_FAR : PC_GATHERED, false);
            else if (LANES == 32 && gather_once(p)) TK_PC_FP8_LAUNCH(LANES == 32 ? PC_GATHERED_ONCE : PC_GATHERED, false);
            else if ((int64_t)p.M * p.K <= kPcThrough) TK_PC_FP8_LAUNCH(PC_GATHERED, true);
            else TK_PC_FP8_LAUNCH(PC_GATHERED, false);
#undef TK_PC_FP8_LAUNCH
            return;
        }
    }
    p.tiles_k = (p.K + LANES * 8 - 1) / (LANES * 8);
    // (token tiles on x, so that successive workgroups write neighbouring pieces of the same transposed rows,
    // measured slower: 19.7 -> 21.1 us transposed, 17.4 -> 20.3 us with SwiGLU)
    const dim3 grid = MODE == PC_E4M3 ? dim3((unsigned)(tiles_m * p.tiles_k)) : dim3((unsigned)p.tiles_k, (unsigned)tiles_m);
#define TK_PC_LAUNCH(T, ...) \
    hipLaunchKernelGGL((per_channel_cast_kernel<MODE, NPT, T, __VA_ARGS__>), grid, block, 0, stream, TK_PC_LAUNCH_ARGS(p))
    if constexpr (MODE == PC_SWIGLU) {
        if (transpose && p.use_clamp) TK_PC_LAUNCH(true, false, LANES, true);
        else if (transpose) TK_PC_LAUNCH(true, false, LANES);
        else if (p.use_clamp) TK_PC_LAUNCH(false, false, LANES, true);
        else TK_PC_LAUNCH(false, false, LANES);
    } else if constexpr (MODE == PC_F32) {   // checked before: no transposed output from fp32
        if (p.pos_to_token) TK_PC_LAUNCH(false, true, LANES);
        else TK_PC_LAUNCH(false, false, LANES);
    } else if (p.pos_to_token) {
        if (transpose) TK_PC_LAUNCH(true, true, LANES);
        else TK_PC_LAUNCH(false, true, LANES);
    } else {
        if (transpose) TK_PC_LAUNCH(true, false, LANES);
        else TK_PC_LAUNCH(false, false, LANES);
    }
#undef TK_PC_LAUNCH
}

template <int MODE, int NPT>
static void launch_per_channel_2(const PerChannelParams &p, bool transpose, hipStream_t stream) {
    const int wide_cols = MODE == PC_E4M3 && !transpose ? 512 : 256;
    const int64_t tiles = (int64_t)((p.M + kPcTileM - 1) / kPcTileM) * ((p.K + wide_cols - 1) / wide_cols);
    bool narrow = tiles < wide_tiles_from<MODE>(transpose, p.pos_to_token != nullptr);
    if (MODE == PC_E4M3 && !transpose && p.pos_to_token && aligned_to(p.x, 16) && aligned_to(p.out, 16))
        narrow = !gather_far(p) && (narrow || gather_repeats(p.num_tokens, p.M));
    if (narrow) launch_per_channel_3<MODE, NPT, 16>(p, transpose, stream);
    else launch_per_channel_3<MODE, NPT, 32>(p, transpose, stream);
}

template <int MODE>
static hipError_t launch_per_channel(const PerChannelParams &p, int num_per_tokens, bool transpose, hipStream_t stream) {
    if (num_per_tokens == 128) launch_per_channel_2<MODE, 128>(p, transpose, stream);
    else launch_per_channel_2<MODE, 32>(p, transpose, stream);
    return hipGetLastError();
}

}  // namespace tk

using namespace tk;

extern "C" int tk_check_per_channel_cast(const void *x, int x_dtype, const float *x_sf, int64_t num_tokens, int64_t K,
                                         const int32_t *pos_to_token, int64_t M, const void *out, const float *out_sf,
                                         int num_per_tokens, int round_sf, int transpose, int swiglu, int use_clamp,
                                         float clamp) {
    (void)round_sf;
    (void)pos_to_token;
    (void)transpose;
    if (x_dtype != TK_BF16 && x_dtype != TK_F32) return TK_ERR_BAD_DTYPE;
    if (x_dtype == TK_F32 && (x_sf || swiglu || transpose)) return TK_ERR_BAD_DTYPE;   // as the reference: plain and gathered casts only
    if (num_per_tokens != 32 && num_per_tokens != 128) return TK_ERR_BAD_GROUP;
    if (num_tokens < 0 || M < 0 || K <= 0 || K % 8 != 0 || M % 16 != 0) return TK_ERR_BAD_SHAPE;
    if (x_sf && (K % 128 != 0 || swiglu)) return TK_ERR_BAD_MODE;
    if (!pos_to_token && num_tokens < M) return TK_ERR_BAD_SHAPE;
    // gathered rows with a negative index are read from row 0 and zeroed by value, so that row must exist
    if (pos_to_token && num_tokens == 0 && M > 0) return TK_ERR_BAD_SHAPE;
    if (swiglu && pos_to_token) return TK_ERR_BAD_MODE;
    if (use_clamp && (!swiglu || !(clamp == clamp))) return TK_ERR_BAD_VALUE;
    if (num_tokens > INT32_MAX - 256 || M > INT32_MAX - 256 || K > (INT32_MAX - 1024) / 2) return TK_ERR_TOO_LARGE;
    if (M == 0) return TK_OK;
    if (!x || !out || !out_sf) return TK_ERR_NULL_POINTER;
    if (!aligned_to(x, x_sf ? 8 : 16) || !aligned_to(out, transpose ? 16 : 8) || !aligned_to(out_sf, 4) || !aligned_to(x_sf, 4))
        return TK_ERR_MISALIGNED;
    const int64_t tiles = ((M + kPcTileM - 1) / kPcTileM) * ((K + 255) / 256);
    if (tiles > INT32_MAX - 8 || (M + kPcTileM - 1) / kPcTileM > 65535) return TK_ERR_TOO_LARGE;   // token tiles ride on grid.y
    return TK_OK;
}

extern "C" int tk_per_channel_cast(const void *x, int x_dtype, const float *x_sf, int64_t num_tokens, int64_t K,
                                   const int32_t *pos_to_token, int64_t M, void *out, float *out_sf, int num_per_tokens,
                                   int round_sf, int transpose, int swiglu, int use_clamp, float clamp, void *stream) {
    const int rc = tk_check_per_channel_cast(x, x_dtype, x_sf, num_tokens, K, pos_to_token, M, out, out_sf, num_per_tokens,
                                             round_sf, transpose, swiglu, use_clamp, clamp);
    if (rc != TK_OK || M == 0) return rc;
    PerChannelParams p;
    p.x = x;
    p.x_sf = x_sf;
    p.pos_to_token = pos_to_token;
    p.out = static_cast<uint8_t *>(out);
    p.out_sf = out_sf;
    p.num_tokens = (int)num_tokens;
    p.K = (int)K;
    p.M = (int)M;
    p.tiles_k = 0;      // set with the tile width
    p.round_sf = round_sf;
    p.use_clamp = use_clamp;
    p.clamp = clamp;
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipError_t e;
    if (swiglu) e = launch_per_channel<PC_SWIGLU>(p, num_per_tokens, transpose != 0, s);
    else if (x_sf) e = launch_per_channel<PC_E4M3>(p, num_per_tokens, transpose != 0, s);
    else if (x_dtype == TK_F32) e = launch_per_channel<PC_F32>(p, num_per_tokens, false, s);
    else e = launch_per_channel<PC_BF16>(p, num_per_tokens, transpose != 0, s);
    return (int)e;
}
