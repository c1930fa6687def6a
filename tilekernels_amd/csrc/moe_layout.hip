// Expert-major ("fused") MoE layout for gfx950: the mapping between the (token, k) routing list and
// the expanded row order, and the row expansion that feeds the fused SwiGLU op.  Integer / byte
// work, HBM- and latency-bound; no LDS tiling beyond per-wave histograms.
//
// Reference semantics: tile_kernels/moe/get_fused_mapping_kernel.py:24-250,
// tile_kernels/moe/expand_to_fused_kernel.py:16-200, tile_kernels/torch/expand_to_fused.py,
// tile_kernels/moe/reduce_fused_kernel.py:12-135, tile_kernels/torch/reduce_fused.py.
#include <atomic>
#include <algorithm>

#include "tk_device.hpp"
#include "tk_host.hpp"

namespace tk {

// ------------------------------------------------------------------------------------------------
// get_fused_mapping: a stable counting sort of the flat (token, k) list by expert, every expert's
// segment padded to a multiple of `alignment`.  Lists of up to 64 Ki pairs take a single launch of
// several workgroups, longer ones two launches (both further down), the longest, and those of more than 512 experts, three, with no
// grid-wide barrier (a single workgroup doing all of it was measured at 70 us for 32 Ki pairs against 18 us for the three
// launches: one CU cannot absorb the scattered 4-byte stores of the hand-out):
//   count  : each wave histograms its own 256-element slice            -> ws[slice][expert]
//   scan   : one workgroup turns the histograms into exclusive offsets  -> ws[slice][expert], expert_start/end
//   assign : each wave walks its slice again in order and hands out positions
// Positions inside an expert follow the flat index (the reference leaves that order open).
constexpr int kSliceElems = 256;   // elements per wave
constexpr int kMaxExperts = 1024;  // bound on the per-wave LDS histogram

__global__ __launch_bounds__(kThreads) void fused_mapping_count_kernel(const int64_t *topk_idx, int numel, int num_experts,
                                                                       int32_t *ws, int32_t *pos_to_expert, int32_t *pos_to_token,
                                                                       int32_t *pos_to_token_topk, int num_expanded) {
    extern __shared__ int32_t hist[];   // [kWaves][num_experts]
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int slice = blockIdx.x * kWaves + wave;
    int32_t *h = hist + wave * num_experts;
    for (int e = lane; e < num_experts; e += 64) h[e] = 0;
    // padding positions keep -1; the assign launch overwrites the live ones
    // (64 bits: buffers of nearly 2^31 positions plus a stride of all workgroups)
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < num_expanded; i += (int64_t)gridDim.x * kThreads) {
        pos_to_expert[i] = -1;
        pos_to_token[i] = -1;
        pos_to_token_topk[i] = -1;
    }
    __syncthreads();
    const int base = slice * kSliceElems;
    for (int j = lane; j < kSliceElems; j += 64) {
        const int i = base + j;
        if (i < numel) {
            const int64_t e = topk_idx[i];
            if (e >= 0 && e < num_experts) atomicAdd(&h[(int)e], 1);
        }
    }
    __syncthreads();
    if (base < numel)
        for (int e = lane; e < num_experts; e += 64) ws[(int64_t)slice * num_experts + e] = h[e];
}

// Mask of the lanes that hold the same expert id as this lane (ids < 0 match nothing): the ballots
// of every bit of the id, intersected.
__device__ __forceinline__ unsigned long long same_expert_lanes(int e, int expert_bits) {
    unsigned long long peers = __ballot(e >= 0);
    for (int b = 0; b < expert_bits; ++b) {
        const bool bit = (e >> b) & 1;
        const unsigned long long m = __ballot(bit);
        peers &= bit ? m : ~m;
    }
    return peers;
}

// One wave hands out positions to the elements [base, base + 64 * STEPS) of the flat (token, k) list, in order, 64 at
// a time; nx[e] is the next free position of expert e for this wave.  The ids of the whole slice are loaded before the
// first is used: one memory round trip per slice instead of one per 64 elements.
template <int STEPS>
__device__ __forceinline__ void assign_range(const int64_t *topk_idx, int base, int numel, int num_topk, int num_experts,
                                             int expert_bits, int32_t *nx, int32_t *pos_to_expert, int32_t *pos_to_token,
                                             int32_t *pos_to_token_topk, int32_t *token_topk_to_pos, int num_expanded) {
    // pos_to_expert == nullptr: the caller fills that array itself (it is a function of the expert offsets alone)
    const int lane = threadIdx.x & 63;
    const unsigned long long below = (1ull << lane) - 1ull;
    int64_t ids[STEPS];
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        const int i = base + j * 64 + lane;
        ids[j] = topk_idx[i < numel ? i : base];
    }
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        const int i = base + j * 64 + lane;
        if (base + j * 64 >= numel) break;             // wave-uniform
        const int64_t v = ids[j];
        const int e = (i < numel && v >= 0 && v < num_experts) ? (int)v : -1;
        const unsigned long long peers = same_expert_lanes(e, expert_bits);
        int pos = -1;
        if (e >= 0) {
            const int first = nx[e];
            pos = first + __popcll(peers & below);
            __builtin_amdgcn_wave_barrier();          // every peer has read before the last one advances the counter
            if ((peers >> lane) == 1ull) nx[e] = first + __popcll(peers);
        }
        __builtin_amdgcn_wave_barrier();
        if (i < numel) token_topk_to_pos[i] = pos;
        if (pos >= 0 && pos < num_expanded) {
            if (pos_to_expert) pos_to_expert[pos] = e;
            pos_to_token[pos] = i / num_topk;
            pos_to_token_topk[pos] = i;
        }
    }
}

// Inclusive prefix sum over the experts with all 1024 threads of a workgroup (Hillis-Steele on two
// ping-pong buffers); returns the index of the buffer that holds the result.
__device__ __forceinline__ int scan_experts(int32_t (*scan)[kMaxExperts], const int32_t *padded, int num_experts) {
    const int t = threadIdx.x;
    scan[0][t] = t < num_experts ? padded[t] : 0;
    __syncthreads();
    int cur = 0;
    for (int d = 1; d < kMaxExperts; d <<= 1) {
        scan[cur ^ 1][t] = scan[cur][t] + (t >= d ? scan[cur][t - d] : 0);
        cur ^= 1;
        __syncthreads();
    }
    return cur;
}

// One workgroup of 1024 threads.  The slice axis is cut into C = 1024 / num_experts chunks (at least
// one) and thread (c, e) owns chunk c of expert e: it sums its chunk (independent loads, so their
// latencies overlap), the chunk totals are exchanged through LDS, and a second walk over the chunk
// (from L2) writes the exclusive offsets.  Expert starts come from a block-wide prefix sum.
__global__ __launch_bounds__(1024) void fused_mapping_scan_kernel(int32_t *ws, int num_slices, int num_experts, int alignment,
                                                                  int32_t *expert_start, int32_t *expert_end,
                                                                  int32_t *num_tokens_per_expert, int32_t *host_counts) {
    __shared__ int32_t total[1024];          // [chunk][expert], chunks * num_experts <= 1024
    __shared__ int32_t padded[kMaxExperts];
    __shared__ int32_t scan[2][kMaxExperts];
    const int chunks = num_experts >= 1024 ? 1 : 1024 / num_experts;
    const int per = (num_slices + chunks - 1) / chunks;
    const int c = threadIdx.x / num_experts, e = threadIdx.x - c * num_experts;
    const bool active = c < chunks;
    const int s0 = c * per, s1 = min(s0 + per, num_slices);

    if (active) {
        int32_t sum = 0;
#pragma unroll 8
        for (int s = s0; s < s1; ++s) sum += ws[(int64_t)s * num_experts + e];
        total[c * num_experts + e] = sum;
    }
    __syncthreads();
    int32_t run = 0;
    if (active) {
        for (int k = 0; k < c; ++k) run += total[k * num_experts + e];
        if (c == 0) {
            int32_t all = 0;
            for (int k = 0; k < chunks; ++k) all += total[k * num_experts + e];
            padded[e] = (all + alignment - 1) / alignment * alignment;
        }
#pragma unroll 8
        for (int s = s0; s < s1; ++s) {
            const int64_t at = (int64_t)s * num_experts + e;
            const int32_t n = ws[at];
            ws[at] = run;          // exclusive offset of this slice inside the expert
            run += n;
        }
    }
    __syncthreads();
    const int cur = scan_experts(scan, padded, num_experts);
    const int t = threadIdx.x;
    if (t < num_experts) {
        const int32_t end = scan[cur][t];
        expert_start[t] = end - padded[t];
        expert_end[t] = end;
        num_tokens_per_expert[t] = padded[t];
        if (host_counts) st_stream4(host_counts + t, (uint32_t)padded[t]);
    }
}

// Row b of the table: how many of the entries 1024 b .. 1024 b + 1023 each expert has.
__global__ __launch_bounds__(kThreads) void fused_mapping_table_kernel(const int64_t *topk_idx, int numel, int num_experts, int32_t *table) {
    extern __shared__ int32_t hist[];   // [num_experts]
    constexpr int U = 1024 / kThreads;
    const int base = blockIdx.x * 1024;
    int64_t ids[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
        const int i = base + j * kThreads + (int)threadIdx.x;
        ids[j] = topk_idx[i < numel ? i : base];
    }
    for (int e = threadIdx.x; e < num_experts; e += kThreads) hist[e] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < U; ++j)
        if (base + j * kThreads + (int)threadIdx.x < numel && ids[j] >= 0 && ids[j] < num_experts) atomicAdd(&hist[(int)ids[j]], 1);
    __syncthreads();
    for (int e = threadIdx.x; e < num_experts; e += kThreads) table[(int64_t)blockIdx.x * num_experts + e] = hist[e];
}

// The whole mapping in one launch, for lists of up to kSingleLaunchPairs (token, k) pairs: no launch has to wait for
// another, and no table in global memory is needed.  A workgroup of 16 waves owns 16 consecutive slices of 64, and instead
// of being told how many entries of every expert precede them it counts them itself: every workgroup reads the whole
// list once (a few hundred KB that stay in the L2) into LDS histograms: all entries, the entries before its own
// range, and one per slice of its own.  From these every workgroup derives the same expert offsets (a prefix sum over
// the padded expert sizes) and its slices' first positions, hands out positions exactly as the assign launch does, and
// marks its share of the padding positions: the ends of the experts e = workgroup, workgroup + gridDim, ... and its
// stride of the unused tail of the buffers.  Measured on MI355X for 4096 tokens, top-8 of 256 experts: 8.0 us, of which
// about half is the counting pass (its LDS atomics), against 17.8 us for the three launches.
constexpr int kSingleLaunchPairs = 64 * 1024 - 1;
constexpr int kSingleWaves = 16;
constexpr int kSingleSlice = 64;            // entries a wave hands out: 1024 per workgroup, so that the scattered stores of the
                                            // hand-out spread over many CUs (256 per wave, 8 workgroups for 32 Ki pairs: 13.6 us)
constexpr int kSingleMaxExperts = 512;      // (1 + kSingleWaves) histograms of 4-byte counters must fit the LDS of a workgroup

// TABLE: longer lists, in two launches.  fused_mapping_table_kernel counts the entries of every 1024 into one row of a table, and
// the workgroups of this kernel sum the table's columns (all rows, and the rows before their own) in place of reading the list.
// What the three launches spent their time on is the scan in the middle: one workgroup, two walks over a table with a row per
// 256 entries, 8.3 of 20 us for 172160 pairs.  A workgroup reads the whole table here, so the table is held short: see
// table_mapping_pays.
template <bool TABLE>
__global__ __launch_bounds__(64 * kSingleWaves) void fused_mapping_single_kernel(const int64_t *topk_idx, int numel, int num_topk,
                                                                                int num_experts, int expert_bits, int alignment,
                                                                                int32_t *pos_to_expert, int32_t *pos_to_token,
                                                                                int32_t *pos_to_token_topk, int32_t *token_topk_to_pos,
                                                                                int32_t *expert_start, int32_t *expert_end,
                                                                                int32_t *num_tokens_per_expert, int num_expanded,
                                                                                const int32_t *table, int32_t *host_counts) {
    // counts[e]: entries of expert e in the whole list (low half) and before this workgroup's range (high half): one
    // LDS atomic per entry for both, which is what this pass spends its time on (a list of fewer than 64 Ki pairs
    // cannot overflow a half; TABLE: two words); slice[w][e]: entries of expert e in slice w of the workgroup's own range
    extern __shared__ int32_t hist[];        // counts[E] (TABLE: all[E], before[E]), slice[kSingleWaves][E]
    __shared__ int32_t padded[kSingleMaxExperts];
    __shared__ int32_t ends[kSingleMaxExperts];
    __shared__ int32_t wave_total[kSingleMaxExperts / 64];
    uint32_t *counts = reinterpret_cast<uint32_t *>(hist);
    constexpr int kCounts = TABLE ? 2 : 1;
    int32_t *slice = hist + kCounts * num_experts;
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
    const int nthreads = 64 * kSingleWaves;
    const int own_base = blockIdx.x * (kSingleWaves * kSingleSlice), own_end = own_base + kSingleWaves * kSingleSlice;

    auto all_of = [&](int e) { return (int32_t)(TABLE ? counts[e] : counts[e] & 0xFFFFu); };
    auto before_of = [&](int e) { return (int32_t)(TABLE ? counts[num_experts + e] : counts[e] >> 16); };

    for (int i = tid; i < (kCounts + kSingleWaves) * num_experts; i += nthreads) hist[i] = 0;
    __syncthreads();
    if constexpr (TABLE) {
        static_assert(kSingleSlice == 64, "one entry per thread");
        const int i = own_base + tid;
        const int64_t v = topk_idx[i < numel ? i : 0];
        // threads beyond the last whole table row of the 1024 words idle; the others read consecutive words
        const int lead = nthreads / num_experts * num_experts, words = (int)gridDim.x * num_experts, own_word = (int)blockIdx.x * num_experts;
        if (tid < lead) {
            int32_t all = 0, before = 0;
#pragma unroll 8
            for (int w = tid; w < words; w += lead) {
                const int32_t n = table[w];
                all += n;
                before += w < own_word ? n : 0;
            }
            const int e = tid % num_experts;
            if (all) atomicAdd(&hist[e], all);
            if (before) atomicAdd(&hist[num_experts + e], before);
        }
        if (i < numel && v >= 0 && v < num_experts) atomicAdd(&slice[wave * num_experts + (int)v], 1);
    }
    auto count = [&](int i, int64_t v) {
        if (v >= 0 && v < num_experts) {
            const int e = (int)v;
            atomicAdd(&counts[e], i < own_base ? 0x10001u : 1u);
            if (i >= own_base && i < own_end) atomicAdd(&slice[((i - own_base) / kSingleSlice) * num_experts + e], 1);
        }
    };
    // The list is read in 16-byte pieces (two ids), 4 of them per thread in flight at a time.  A thread's loads beyond the end of the
    // list read its first piece, and in a short list nearly all of them are beyond it: with 16 in flight, us for 512 / 2720 / 8000 /
    // 32768 pairs: 5.06 / 5.31 / 5.70 / 8.67; 4: 3.65 / 3.93 / 4.40 / 8.01; 2: 3.47 / 3.79 / 4.39 / 8.26; 1: 3.49 / 3.86 / 4.50 / 8.81.
    const int head = TABLE ? 0 : (int)((reinterpret_cast<uintptr_t>(topk_idx) >> 3) & 1);      // ids before the first 16-byte boundary
    const int pairs = TABLE ? 0 : (numel - head) / 2;
    const u32x4 *wide = reinterpret_cast<const u32x4 *>(topk_idx + head);
    constexpr int U = 4;
    for (int p0 = 0; p0 < pairs; p0 += U * nthreads) {
        u32x4 w[U];
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int pi = p0 + j * nthreads + tid;
            w[j] = wide[pi < pairs ? pi : 0];
            vmem_issue_gap();
        }
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int pi = p0 + j * nthreads + tid;
            if (pi < pairs) {
                count(head + 2 * pi, (int64_t)(((uint64_t)w[j].y << 32) | w[j].x));
                count(head + 2 * pi + 1, (int64_t)(((uint64_t)w[j].w << 32) | w[j].z));
            }
        }
    }
    if (tid == 0 && head) count(0, topk_idx[0]);
    if (!TABLE && tid == 1 && head + 2 * pairs < numel) count(numel - 1, topk_idx[numel - 1]);
    __syncthreads();
    // prefix sum over the padded expert sizes: inside each wave by shuffles, across the (at most 8) waves through LDS
    int32_t mine = 0, incl = 0;
    if (tid < kSingleMaxExperts) {
        mine = tid < num_experts ? (int32_t)(((uint32_t)all_of(tid) + alignment - 1) / alignment * alignment) : 0;
        if (host_counts && blockIdx.x == 0 && tid < num_experts) st_stream4(host_counts + tid, (uint32_t)mine);
        incl = mine;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int32_t up = __shfl_up(incl, d, 64);
            if (lane >= d) incl += up;
        }
        if (lane == 63) wave_total[wave] = incl;
    }
    __syncthreads();
    if (tid < num_experts) {
        int32_t offset = 0;
        for (int w = 0; w < wave; ++w) offset += wave_total[w];
        const int32_t end = offset + incl, start = end - mine;
        padded[tid] = mine;
        ends[tid] = end;
        if (blockIdx.x == 0) {
            expert_start[tid] = start;
            expert_end[tid] = end;
            num_tokens_per_expert[tid] = mine;
        }
        // first position of every slice of this workgroup inside the expert
        int32_t run = start + before_of(tid);
        for (int w = 0; w < kSingleWaves; ++w) {
            const int32_t n = slice[w * num_experts + tid];
            slice[w * num_experts + tid] = run;
            run += n;
        }
    }
    __syncthreads();
    const int total = ends[num_experts - 1];
    const int base = own_base + wave * kSingleSlice;
    if (base < numel)
        assign_range<kSingleSlice / 64>(topk_idx, base, numel, num_topk, num_experts, expert_bits, slice + wave * num_experts, nullptr,
                                        pos_to_token, pos_to_token_topk, token_topk_to_pos, num_expanded);
    if constexpr (TABLE) {
        // Every position's expert by bisection of the ends, and the padding marks, in one stride over the buffers.
        for (int64_t i = (int)blockIdx.x * nthreads + tid; i < num_expanded; i += (int)gridDim.x * nthreads) {
            int lo = 0, hi = num_experts - 1;              // the first expert that ends behind i (experts without entries end where they start)
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (ends[mid] > i) hi = mid;
                else lo = mid + 1;
            }
            const bool live = i < total && i < ends[lo] - padded[lo] + all_of(lo);
            pos_to_expert[i] = live ? lo : -1;
            if (!live) {
                pos_to_token[i] = -1;
                pos_to_token_topk[i] = -1;
            }
        }
        return;
    }
    // The experts this workgroup looks after, a wave per expert: pos_to_expert of the whole segment (it follows from the
    // offsets, and written here it leaves as whole lines instead of one scattered word per entry: the hand-out above
    // is bound by the rate at which one CU issues scattered stores) and the padding marks at the segment's end.
    for (int e = (int)blockIdx.x + wave * (int)gridDim.x; e < num_experts; e += kSingleWaves * (int)gridDim.x) {
        const int end = ends[e], start = end - padded[e], first = start + all_of(e);
        for (int i = start + lane; i < end && i < num_expanded; i += 64) pos_to_expert[i] = i < first ? e : -1;
        for (int i = first + lane; i < end && i < num_expanded; i += 64) {
            pos_to_token[i] = -1;
            pos_to_token_topk[i] = -1;
        }
    }
    // positions beyond the last expert
    for (int64_t i = (int64_t)total + (int)blockIdx.x * nthreads + tid; i < num_expanded; i += (int)gridDim.x * nthreads) {      // (64 bits: as in the count kernel)
        pos_to_expert[i] = -1;
        pos_to_token[i] = -1;
        pos_to_token_topk[i] = -1;
    }
}

__global__ __launch_bounds__(kThreads) void fused_mapping_assign_kernel(const int64_t *topk_idx, int numel, int num_topk,
                                                                        int num_experts, int expert_bits, const int32_t *ws,
                                                                        const int32_t *expert_start, int32_t *pos_to_expert,
                                                                        int32_t *pos_to_token, int32_t *pos_to_token_topk,
                                                                        int32_t *token_topk_to_pos, int num_expanded) {
    extern __shared__ int32_t next[];   // [kWaves][num_experts]: next free position per expert, per wave
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int slice = blockIdx.x * kWaves + wave;
    const int base = slice * kSliceElems;
    if (base >= numel) return;          // whole wave; no barrier below
    int32_t *nx = next + wave * num_experts;
    for (int e = lane; e < num_experts; e += 64) nx[e] = expert_start[e] + ws[(int64_t)slice * num_experts + e];
    __builtin_amdgcn_wave_barrier();
    assign_range<kSliceElems / 64>(topk_idx, base, numel, num_topk, num_experts, expert_bits, nx, pos_to_expert, pos_to_token,
                                   pos_to_token_topk, token_topk_to_pos, num_expanded);
}

// ------------------------------------------------------------------------------------------------
// expand_to_fused.  Rows are moved as raw 16-byte pieces, so any element type works; optional 4-byte
// scale rows travel the same way into a row-major or column-major scale tensor.
//
// One load and one store per thread.  What bounds this operator is the write stream (8 bytes written
// per byte read at top-8), and on MI355X that stream runs the faster the fewer stores a thread issues:
// filling 268 MB takes 40.6 us with one 16-byte store per thread, 44 us with 2 or 4, 47 us with 8 and
// 53 us with 16.  A workgroup therefore copies one 4 KB chunk of one token's row to ONE of its
// positions, and the row is read once per position instead of once: the re-reads hit the L2, because
// workgroups are dealt to the 8 XCDs (one L2 each) round-robin and the workgroups of a chunk are
// numbered 8 apart, which puts all of them on one XCD back to back.  (Measured for [4096, 4096] bf16,
// top-8, random positions, 268 MB written: 50.6 us this way, 57 us with the copies of a chunk on
// different XCDs, 61 us with one load and 8 stores per thread.)
// The workgroups after those each look at a few consecutive expanded rows (8 KB worth) and zero the ones
// that are padding.
constexpr int kExpandChunk = kThreads * 16;

// Non-temporal 16-byte stores: writing the same 268 MB as whole 8 KB rows per wave takes 52 us with them and
// 62 us with plain stores; pairs of 8-byte system-scope stores are several times slower still.
__device__ __forceinline__ void expand_store16(void *p, u32x4 v) { __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(p)); }

// Padding workgroup `pb` of the short-rows kernel: zero the rows among its pad_rows consecutive expanded rows that no
// token maps to (the same loop as in the kernel for long rows, which keeps its own copy: sharing this function cost
// that kernel 2 % with scale rows).
__device__ __forceinline__ void expand_zero_padding(int pb, int pad_rows, int num_expanded, int64_t row_bytes, uint8_t *out,
                                                    const int32_t *pos_to_expert, bool with_sf, int sf_cols, uint32_t *out_sf,
                                                    int64_t out_sf_ld, int sf_col_major) {
    const int r0 = pb * pad_rows;
    for (int r = r0; r < r0 + pad_rows && r < num_expanded; ++r) {
        if (uniform_load(pos_to_expert + r) >= 0) continue;
        uint8_t *dst = out + (int64_t)r * row_bytes;
        for (int64_t off = (int64_t)threadIdx.x * 16; off < row_bytes; off += kExpandChunk) expand_store16(dst + off, u32x4{0u, 0u, 0u, 0u});
        if (with_sf)
            for (int j = threadIdx.x; j < sf_cols; j += kThreads) out_sf[sf_col_major ? (int64_t)j * out_sf_ld + r : (int64_t)r * out_sf_ld + j] = 0u;
    }
}

// EVERY: a workgroup per list entry, one store per thread, as described above.  That pays for full lists that fill
// a long buffer.  Otherwise one workgroup serves every live entry of a token's chunk: it reads the list with one load per lane, a
// ballot says which entries have a position, and there is one store per thread for each of them.  What bounds an
// expert-parallel rank's expansion with EVERY is the dispatch of workgroups that find no position (0.7 ns each, whatever
// they do).  us per call on MI355X, EVERY / one per token (codes with scales, top-8 unless said):
//   one of 8 ranks: 21504 tokens -> [24064, 7168]  214 / 59.5      340 tokens -> [6784, 4096] (worst-case buffer)  6.7 / 5.4
//   full lists: [512, 4096] -> [5120]  6.6 / 4.7      [2048, 7168] -> [17536]  31.3 / 27.9      top-2 of [8192, 7168]  32.1 / 29.5
//   with much padding, top-2: bf16 [3000, 2560] -> [8192]  12.9 / 10.4, codes [10000, 7168] -> [30000]  43.2 / 44.2; worst-case buffers of one of
//   8 ranks, bf16 [3000, 2560] -> [9984]  15.0 / 10.7, [5000, 7168] -> [13952]  56.2 / 44.1
//   bf16 -> rows of 4096, 110 MB 25.6 / 22.8, 132 MB 30.3 / 27.2, 154 MB 35.4 / 32.9, 184 MB 42.0 / 40.2, 203 MB 46.4 / 48.1, 234 MB 53.2 / 54.5,
//   304 MB 68.3 / 70.6, 404 MB 90.9 / 95.4 (2048 and codes of 4096 the same);  7168, 168 MB 38.3 / 35.6, 236 MB 54.6 / 51.0, 407 MB 92.5 / 89.9;
//   a third of [48128] rows of 4096 padding: codes with scales, 197 MB 38.1 / 39.2, bf16, 394 MB 64.4 / 73.5
// The line lies at 160 MB for all of them, so that no output beyond it is slower than entry by entry.
// SF: there are scales (with EVERY there may be); otherwise nothing of them is looked at.
template <bool EVERY, bool SF>
__global__ __launch_bounds__(kThreads) void expand_to_fused_kernel(const uint8_t *x, int64_t row_bytes, const int32_t *token_topk_to_pos,
                                                                   int num_topk, int chunks, int copy_blocks, int num_tokens,
                                                                   int num_expanded, uint8_t *out, const int32_t *pos_to_expert,
                                                                   const uint32_t *x_sf, int sf_cols, uint32_t *out_sf,
                                                                   int64_t out_sf_ld, int sf_col_major, int pad_rows) {
    const int b = blockIdx.x;
    if (b < copy_blocks) {
        // b = 8 * ((token group * chunks + chunk) * entries + entry) + token within its group of 8
        const int q = b >> 3;
        const int k = EVERY ? q % num_topk : 0, q2 = EVERY ? q / num_topk : q;
        const int c = q2 % chunks, t = (q2 / chunks) * 8 + (b & 7);
        if (t >= num_tokens) return;
        const int64_t off = (int64_t)c * kExpandChunk + threadIdx.x * 16;
        const u32x4 *src = reinterpret_cast<const u32x4 *>(x + (int64_t)t * row_bytes + off);
        const int32_t *list = token_topk_to_pos + (int64_t)t * num_topk;
        u32x4 v = u32x4{0u, 0u, 0u, 0u};
        if constexpr (EVERY) {
            const int p = uniform_load(list + k);
            if (off < row_bytes) v = *src;   // cached: read num_topk times
            if (p < 0 || p >= num_expanded) return;
            if (off < row_bytes) expand_store16(out + (int64_t)p * row_bytes + off, v);
            if (x_sf && c == 0)
                for (int j = threadIdx.x; j < sf_cols; j += kThreads)
                    out_sf[sf_col_major ? (int64_t)j * out_sf_ld + p : (int64_t)p * out_sf_ld + j] = x_sf[(int64_t)t * sf_cols + j];
            return;
        }
        // The thread's first scale word is loaded once, with the row: loaded at each copy it is waited for at each copy.  Where its copies go is
        // worked out behind the ballot, once there is one: in front of it a workgroup without a position did all of that, too (codes with
        // scales, one of 8 ranks, us: top-1 of [8192, 2048] 5.8 / 5.1, [21504, 2048] 11.4 / 9.8, top-2 of [8192, 7168] 13.3 / 12.6).
        uint32_t sf0 = 0;
        for (int k0 = 0; k0 < num_topk; k0 += 64) {
            const int kk = k0 + (threadIdx.x & 63);
            const int pos = list[kk < num_topk ? kk : 0];
            if (k0 == 0) {      // a token without any position is rare: not waited for
                if (off < row_bytes) v = *src;
                if (SF && c == 0) sf0 = x_sf[(int64_t)t * sf_cols + ((int)threadIdx.x < sf_cols ? threadIdx.x : 0)];
            }
            unsigned long long live = __builtin_amdgcn_ballot_w64(kk < num_topk && pos >= 0 && pos < num_expanded);
            if (!live) continue;
            int i = threadIdx.x, token = t, turned = sf_col_major;
            if constexpr (SF) asm volatile("" : "+v"(i), "+s"(token), "+s"(turned));      // (opaque, or the compiler computes all of this in front of the loop)
            const bool scales = SF && c == 0, scale_word = scales && i < sf_cols;
            const uint32_t *sf_row = x_sf + (int64_t)token * sf_cols;
            const int64_t sf_step = turned ? 1 : out_sf_ld, sf_word = turned ? out_sf_ld : 1;
            uint32_t *sf_dst = out_sf + (int64_t)i * sf_word;
            for (; live; live &= live - 1) {
                const int64_t p = __builtin_amdgcn_readlane(pos, __builtin_ctzll(live));
                if (off < row_bytes) expand_store16(out + p * row_bytes + off, v);
                if (scale_word) sf_dst[p * sf_step] = sf0;
                if (scales && sf_cols > kThreads)
                    for (int j = i + kThreads; j < sf_cols; j += kThreads) out_sf[j * sf_word + p * sf_step] = sf_row[j];
            }
        }
    } else {
        const int r0 = (b - copy_blocks) * pad_rows;
        for (int r = r0; r < r0 + pad_rows && r < num_expanded; ++r) {
            if (uniform_load(pos_to_expert + r) >= 0) continue;
            uint8_t *dst = out + (int64_t)r * row_bytes;
            for (int64_t off = (int64_t)threadIdx.x * 16; off < row_bytes; off += kExpandChunk) expand_store16(dst + off, u32x4{0u, 0u, 0u, 0u});
            if (x_sf)
                for (int j = threadIdx.x; j < sf_cols; j += kThreads) out_sf[sf_col_major ? (int64_t)j * out_sf_ld + r : (int64_t)r * out_sf_ld + j] = 0u;
        }
    }
}

// Rows of at most 2 KB (a kernel of its own: as a branch of the one above it cost that one 5 %).  The workgroup's
// threads form kpw groups of tpr threads (tpr * 16 >= row_bytes), and group g copies the row to position kg * kpw + g
// of the token, still one load and one store per thread.  (With one position per workgroup half or more of the
// threads had nothing to copy: bf16 [32768, 1024], top-8: 198.7 us, 124.6 us this way.)
// EVERY as above; without it kpw counts tokens, and group g serves all entries of token b * kpw + g (us, EVERY / per token:
// codes [21504, 1280] of 8 ranks 47 / 17.5; top-8 of [8192, 1024] codes 26.2 / 24.8; of bf16 [32768, 1024] 133.5 / 138.9).
template <bool EVERY, bool SF>
__global__ __launch_bounds__(kThreads) void expand_short_rows_kernel(const uint8_t *x, int64_t row_bytes, const int32_t *token_topk_to_pos,
                                                                     int num_topk, int kpw, int tpr, int copy_blocks, int num_tokens,
                                                                     int num_expanded, uint8_t *out, const int32_t *pos_to_expert,
                                                                     const uint32_t *x_sf, int sf_cols, uint32_t *out_sf,
                                                                     int64_t out_sf_ld, int sf_col_major, int pad_rows) {
    const int b = blockIdx.x;
    if (b < copy_blocks) {
        const int g = (int)threadIdx.x / tpr, i = (int)threadIdx.x - g * tpr;
        const int64_t off = (int64_t)i * 16;
        int k = 0, t;
        if (EVERY) {
            // b = 8 * ((token group * groups of positions) + kg) + token within its group of 8
            const int kgroups = (num_topk + kpw - 1) / kpw;
            const int q = b >> 3;
            k = (q % kgroups) * kpw + g;
            t = (q / kgroups) * 8 + (b & 7);
        } else {
            t = b * kpw + g;
        }
        if (t >= num_tokens || g >= kpw || k >= num_topk) return;
        const u32x4 *src = reinterpret_cast<const u32x4 *>(x + (int64_t)t * row_bytes + off);
        const int32_t *list = token_topk_to_pos + (int64_t)t * num_topk;
        u32x4 v = u32x4{0u, 0u, 0u, 0u};
        if constexpr (EVERY) {
            const int p = list[k];
            if (off < row_bytes) v = *src;   // cached: read num_topk times
            if (p < 0 || p >= num_expanded) return;
            if (off < row_bytes) expand_store16(out + (int64_t)p * row_bytes + off, v);
            if (x_sf)
                for (int j = i; j < sf_cols; j += tpr)
                    out_sf[sf_col_major ? (int64_t)j * out_sf_ld + p : (int64_t)p * out_sf_ld + j] = x_sf[(int64_t)t * sf_cols + j];
            return;
        }
        if (off < row_bytes) v = *src;
        uint32_t sf0 = 0;
        if (SF) sf0 = x_sf[(int64_t)t * sf_cols + (i < sf_cols ? i : 0)];
        for (int k0 = 0; k0 < num_topk; k0 += 8) {
            int p[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) p[j] = list[k0 + j < num_topk ? k0 + j : k0];
            bool live = false;
#pragma unroll
            for (int j = 0; j < 8; ++j) live |= (unsigned)p[j] < (unsigned)num_expanded;
            if (!live) continue;
            // (as in expand_to_fused_kernel)
            int word = i, token = t, turned = sf_col_major;
            if constexpr (SF) asm volatile("" : "+v"(word), "+v"(token), "+s"(turned));
            const bool scale_word = SF && word < sf_cols;
            const uint32_t *sf_row = x_sf + (int64_t)token * sf_cols;
            const int64_t sf_step = turned ? 1 : out_sf_ld, sf_word = turned ? out_sf_ld : 1;
            uint32_t *sf_dst = out_sf + (int64_t)word * sf_word;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (k0 + j >= num_topk || (unsigned)p[j] >= (unsigned)num_expanded) continue;
                if (off < row_bytes) expand_store16(out + (int64_t)p[j] * row_bytes + off, v);
                if (scale_word) sf_dst[p[j] * sf_step] = sf0;
                if (SF && sf_cols > tpr)
                    for (int w = word + tpr; w < sf_cols; w += tpr) out_sf[w * sf_word + p[j] * sf_step] = sf_row[w];
            }
        }
    } else {
        expand_zero_padding(b - copy_blocks, pad_rows, num_expanded, row_bytes, out, pos_to_expert, x_sf != nullptr, sf_cols, out_sf, out_sf_ld,
                            sf_col_major);
    }
}

// ------------------------------------------------------------------------------------------------
// reduce_fused: the inverse of the expansion.  out[t] = sum over k of x[pos(t, k)] * s(t, k), accumulated in fp32 with
// one fused multiply-add per term, in the order k = 0, 1, ... (so that results are reproducible bit for bit), where
// s = topk_weights[t, k] (or 1) times x_sf[pos] (if given); positions < 0 are skipped.  The sum is scaled by *sf (if
// given) and rounded to the output type.
//
// What bounds it is the gather of whole rows from HBM.  A wave owns 512 columns of one token and asks for all its terms' pieces, up to
// 8, before it uses the first.  Positions, weights and scales are the same for the whole wave and come through the scalar path.  A
// rank of an expert-parallel group holds few of a token's experts, one or two of eight on average, and a term that is not live must
// cost nothing: place-holders for it (row 0, so that there is no branch around a load) take as long as rows.  So a group of terms
// that are all live loads without a branch, any other skips its dead terms by branches between the loads; that works because the
// loads' addresses are buffers in scalar registers (see reduce_load).
// us on MI355X, place-holders / live terms found by a ballot over positions that a vector load fetched, 512 columns of 4 tokens or
// 1024 of 2 per workgroup / this, all with weights:
//   bf16 1 of 8 live: [21537, 1280] -> [20000, 1280] 34.5 / 21.3 / 18.9;  [4096, 7168] into a worst-case buffer 40.5 / 21.3 / 19.7
//   bf16 8 of 8: [4096, 512] 7.05 / 7.1 / 7.05;  [.., 1280] 15.9 / 17.0 / 16.1;  [.., 2048] 25.2 / 25.9 / 25.2;  [.., 2560] 35.3 / 31.4 / 31.1;
//   [.., 4096] 50.1 / 49.2 / 49.2;  [.., 7168] 88.6 / 86.3 / 85.6;  340 tokens of 4096 5.07 / 5.4 / 5.1;  [8192, 1280], 2 of 2: 10.8 / 12.6 / 11.2
//   fp32 8 of 8: [4096, 1280] 37.8 / 39.2 / 36.4;  [.., 2048] 50.5 / 51.2 / 50.2;  [.., 4096] 103.2 / 104.0 / 100.3;  64 tokens of 7168 4.1 / 4.9 / 4.2
// fp32 rows whose length is a multiple of 512: a thread's 8 elements are two runs of 4, 256 columns apart, so that each
// of its 16-byte loads (and of its fp32 stores) is, over the wave, 1024 consecutive bytes.  With the 8 elements in one
// run, every instruction touches half of each cache line it names (fp32 [81792, 4096] -> fp32, top-8: 220 instead of 210 us).
struct SplitF32 {};
template <typename InT> struct ReduceIn;
template <> struct ReduceIn<bf16_t> { typedef Raw8<bf16_t> raw; typedef bf16_t elem; static constexpr int lane_bytes = 16, second = 0; };
template <> struct ReduceIn<float> { typedef Raw8<float> raw; typedef float elem; static constexpr int lane_bytes = 32, second = 16; };
template <> struct ReduceIn<SplitF32> { typedef Raw8<float> raw; typedef float elem; static constexpr int lane_bytes = 16, second = 1024; };

// One lane's 8 elements of a piece of 512 columns.  The piece is a buffer of its own, `bytes` long: lanes beyond the end of the row
// read zeros and touch no memory, and no register of the lane holds an address (with addresses in registers a load behind a branch
// waits for an earlier one whose target the address is formed in).
template <typename InT>
__device__ __forceinline__ void reduce_load(typename ReduceIn<InT>::raw &raw, const uint8_t *piece, uint32_t bytes, uint32_t lane_off) {
    const __amdgpu_buffer_rsrc_t buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(piece), 0, (int)bytes, 0x00020000);
    constexpr int kNonTemporal = 2;
    const auto at = [&](uint32_t off) { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(buf, off, 0, kNonTemporal)); };
    if constexpr (ReduceIn<InT>::second != 0) {
        raw.a = at(lane_off);
        vmem_issue_gap();
        raw.b = at(lane_off + ReduceIn<InT>::second);
    } else {
        raw.w = at(lane_off);
    }
    vmem_issue_gap();
}

// U consecutive terms of a token, those in `live` only (ALL: every one).  Everything but the pieces comes through the scalar path.
template <typename InT, int U, bool ALL>
__device__ __forceinline__ void reduce_terms(float (&acc)[8], const uint8_t *x, uint32_t bytes, uint32_t lane_off, uint64_t row_bytes, uint32_t num_expanded,
                                             const uint32_t (&pos)[U], const float *weights, const float *x_sf, int left = U) {
    typename ReduceIn<InT>::raw raw[U];
    uint32_t live = 0;
    float w[U], f[U];
#pragma unroll
    for (int j = 0; j < U; ++j)
        if (ALL || pos[j] < num_expanded) {
            live |= 1u << j;
            reduce_load<InT>(raw[j], x + pos[j] * row_bytes, bytes, lane_off);
        }
    if constexpr (!ALL) {
        // (behind this the compiler no longer knows that the conditions below are those above: it would sink each load to its use)
        live = (uint32_t)__builtin_amdgcn_readfirstlane((int)live);
        asm volatile("" : "+s"(live));
    }
#pragma unroll
    for (int j = 0; j < U; ++j) w[j] = f[j] = 1.0f;
    if (weights) {
#pragma unroll
        for (int j = 0; j < U; ++j) w[j] = uniform_load(weights + (ALL ? j : min(j, left - 1)));
    }
    if (x_sf) {
#pragma unroll
        for (int j = 0; j < U; ++j) f[j] = uniform_load(x_sf + (ALL || pos[j] < num_expanded ? pos[j] : 0u));
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < U; ++j) {
        if (!ALL && !(live >> j & 1)) continue;
        float v[8];
        raw[j].get(v);
        const float s = w[j] * f[j];
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] = __builtin_fmaf(v[i], s, acc[i]);
    }
}

template <typename InT, int U>
__device__ __forceinline__ void reduce_group(float (&acc)[8], const uint8_t *x, uint32_t bytes, uint32_t lane_off, uint64_t row_bytes, uint32_t num_expanded,
                                             const int32_t *list, const float *weights, const float *x_sf) {
    uint32_t pos[U], last = 0;
#pragma unroll
    for (int j = 0; j < U; ++j) pos[j] = (uint32_t)uniform_load(list + j);
    // (written out: the compiler takes the maximum of uniform values through the vector unit)
#pragma unroll
    for (int j = 0; j < U; ++j) asm("s_max_u32 %0, %1, %2" : "=s"(last) : "s"(last), "s"(pos[j]) : "scc");
    if (last < num_expanded) reduce_terms<InT, U, true>(acc, x, bytes, lane_off, row_bytes, num_expanded, pos, weights, x_sf);
    else reduce_terms<InT, U, false>(acc, x, bytes, lane_off, row_bytes, num_expanded, pos, weights, x_sf);
}

// The last five to seven terms.  Of a list with dead terms all live ones together: four and then the rest are two round trips (one of 8
// ranks, 6 terms: bf16 [512, 4096] 3.4 / 3.2 us, [1100, 7168] 7.6 / 7.0, [8192, 4096] 21.0 / 19.8).  A full list is better off in steps, which
// hold fewer loads (6 of 6: bf16 [4500, 2048] 22.5 together / in steps 21.85).
template <typename InT>
__device__ __forceinline__ void reduce_rest(float (&acc)[8], const uint8_t *x, uint32_t bytes, uint32_t lane_off, uint64_t row_bytes, uint32_t num_expanded,
                                            const int32_t *list, const float *weights, const float *x_sf, int left) {
    uint32_t pos[8], last = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) pos[j] = (uint32_t)uniform_load(list + min(j, left - 1));
#pragma unroll
    for (int j = 0; j < 7; ++j) asm("s_max_u32 %0, %1, %2" : "=s"(last) : "s"(last), "s"(pos[j]) : "scc");
    if (last < num_expanded) {
        reduce_terms<InT, 4, true>(acc, x, bytes, lane_off, row_bytes, num_expanded, {pos[0], pos[1], pos[2], pos[3]}, weights, x_sf);
        if (left & 2) reduce_terms<InT, 2, true>(acc, x, bytes, lane_off, row_bytes, num_expanded, {pos[4], pos[5]}, weights ? weights + 4 : weights, x_sf);
        if (left & 1) reduce_terms<InT, 1, true>(acc, x, bytes, lane_off, row_bytes, num_expanded, {pos[7]}, weights ? weights + (left - 1) : weights, x_sf);
    } else {
#pragma unroll
        for (int j = 5; j < 8; ++j)
            if (j >= left) pos[j] = 0xFFFFFFFFu;
        reduce_terms<InT, 8, false>(acc, x, bytes, lane_off, row_bytes, num_expanded, pos, weights, x_sf, left);
    }
}

// OUT: 0 bf16, 1 fp32, 2 E4M3
template <typename InT, int OUT>
__device__ __forceinline__ void reduce_store(const float (&acc)[8], void *out, int64_t idx) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    constexpr bool SPLIT = ReduceIn<InT>::second > 16;
    if (OUT == 1) {
        u32x4 *o = reinterpret_cast<u32x4 *>(reinterpret_cast<float *>(out) + idx);
        __builtin_nontemporal_store(u32x4{f2u(acc[0]), f2u(acc[1]), f2u(acc[2]), f2u(acc[3])}, o);
        __builtin_nontemporal_store(u32x4{f2u(acc[4]), f2u(acc[5]), f2u(acc[6]), f2u(acc[7])}, o + (SPLIT ? 64 : 1));
    } else if (OUT == 0) {
        u32x4 w;
        w.x = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{acc[0], acc[1]}), bf16x2));
        w.y = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{acc[2], acc[3]}), bf16x2));
        w.z = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{acc[4], acc[5]}), bf16x2));
        w.w = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{acc[6], acc[7]}), bf16x2));
        // (written through: bf16 [4096, 4096] from top-8 of 256 experts 50.3 -> 49.2 us on MI355X against a non-temporal
        // store; the stores of most other kernels here lose that way, the expansion 64 -> 110 us)
        st_stream16(reinterpret_cast<uint16_t *>(out) + idx, w);
    } else if (SPLIT) {
        const u32x2 codes = pack_e4m3x8<false>(acc);
        st_stream4(reinterpret_cast<uint8_t *>(out) + idx, codes.x);
        st_stream4(reinterpret_cast<uint8_t *>(out) + idx + 256, codes.y);
    } else {
        st_stream8(reinterpret_cast<uint8_t *>(out) + idx, pack_e4m3x8<false>(acc));
    }
}

// A workgroup takes `side` pieces of one token, or (STACKED, side 1 or 2) those of 4 / side tokens.  FEW: one or two terms.
template <typename InT, int OUT, bool STACKED, bool FEW>
__global__ __launch_bounds__(kThreads) void reduce_fused_kernel(const typename ReduceIn<InT>::elem *x, const int32_t *token_topk_to_pos, int num_tokens,
                                                                int num_topk, int hidden, int num_expanded, int shape,
                                                                const float *topk_weights, const float *x_sf, const float *sf, void *out) {
    constexpr uint32_t kElem = sizeof(typename ReduceIn<InT>::elem);
    const int side = shape & 7, one_col = shape >> 3;
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int t = STACKED ? (tile_grid_row(one_col) << (3 - side)) + (wave >> (side - 1)) : tile_grid_row(one_col);
    const int piece = tile_grid_col(one_col) * side + (STACKED ? wave & (side - 1) : wave);
    if (t >= num_tokens) return;
    const int cols = min(hidden - piece * kStripCols, kStripCols);
    const uint32_t lane_off = (uint32_t)lane * ReduceIn<InT>::lane_bytes;
    const uint8_t *xp = reinterpret_cast<const uint8_t *>(x) + (uint64_t)(uint32_t)piece * (kStripCols * kElem);
    const uint64_t row_bytes = (uint64_t)(uint32_t)hidden * kElem;
    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.0f;
    const int32_t *list = token_topk_to_pos + (int64_t)t * num_topk;
    const float *weights = topk_weights ? topk_weights + (int64_t)t * num_topk : nullptr;
    int left = num_topk;
#define TK_REDUCE_TERMS(U)                                                                                                       \
    do {                                                                                                                         \
        reduce_group<InT, U>(acc, xp, (uint32_t)cols * kElem, lane_off, row_bytes, (uint32_t)num_expanded, list, weights, x_sf); \
        list += U;                                                                                                               \
        if (weights) weights += U;                                                                                               \
    } while (0)
    if constexpr (!FEW) {
        for (; left >= 8; left -= 8) TK_REDUCE_TERMS(8);
        if (left > 4) {
            reduce_rest<InT>(acc, xp, (uint32_t)cols * kElem, lane_off, row_bytes, (uint32_t)num_expanded, list, weights, x_sf, left);
            left = 0;
        }
        if (left & 4) TK_REDUCE_TERMS(4);
    }
    if (left & 2) TK_REDUCE_TERMS(2);
    if (left & 1) TK_REDUCE_TERMS(1);
#undef TK_REDUCE_TERMS
    if (sf) {
        const float f = uniform_load(sf);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] = acc[i] * f;
    }
    // the lane's first column; SPLIT: elements col .. col + 3 and col + 256 .. col + 259 (whole pieces only)
    const int col = piece * kStripCols + lane * (int)(ReduceIn<InT>::lane_bytes / kElem);
    if (col < hidden) reduce_store<InT, OUT>(acc, out, (int64_t)t * hidden + col);
}

// reduce_fused without a single expanded row: every term is skipped, the result is zeros.  (The reduction kernel
// reads the first row's scale in the place of a skipped term's, and there is none then.)
__global__ __launch_bounds__(kThreads) void reduce_zero_kernel(uint64_t *out, int64_t words) {
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < words; i += (int64_t)gridDim.x * kThreads) out[i] = 0ull;
}

}  // namespace tk

using namespace tk;

extern "C" int64_t tk_fused_mapping_workspace_bytes(int64_t num_tokens, int num_topk, int num_experts) {
    if (num_tokens < 0 || num_topk <= 0 || num_experts <= 0) return 0;
    const int64_t slices = (num_tokens * num_topk + kSliceElems - 1) / kSliceElems;
    const int64_t padded = (slices + kWaves - 1) / kWaves * kWaves;       // whole workgroups
    return padded * num_experts * (int64_t)sizeof(int32_t);
}

extern "C" int tk_check_get_fused_mapping(const int64_t *topk_idx, int64_t num_tokens, int num_topk, int num_experts,
                                          int alignment, int64_t num_expanded, const int32_t *pos_to_expert,
                                          const int32_t *pos_to_token, const int32_t *pos_to_token_topk,
                                          const int32_t *token_topk_to_pos, const int32_t *expert_start,
                                          const int32_t *expert_end, const int32_t *num_tokens_per_expert,
                                          const void *workspace, int64_t workspace_bytes) {
    if (num_tokens < 0 || num_topk <= 0 || num_expanded < 0) return TK_ERR_BAD_SHAPE;
    if (num_experts <= 0 || num_experts > kMaxExperts) return TK_ERR_BAD_GROUP;
    if (alignment <= 0) return TK_ERR_BAD_VALUE;
    if (num_tokens * num_topk > INT32_MAX - 1024 || num_expanded > INT32_MAX - 1024) return TK_ERR_TOO_LARGE;
    if (!expert_start || !expert_end || !num_tokens_per_expert) return TK_ERR_NULL_POINTER;
    if (num_tokens > 0 && (!topk_idx || !token_topk_to_pos || !workspace)) return TK_ERR_NULL_POINTER;
    if (num_expanded > 0 && (!pos_to_expert || !pos_to_token || !pos_to_token_topk)) return TK_ERR_NULL_POINTER;
    if (workspace_bytes < tk_fused_mapping_workspace_bytes(num_tokens, num_topk, num_experts)) return TK_ERR_BAD_STRIDE;
    if (!aligned_to(topk_idx, 8) || !aligned_to(workspace, 4)) return TK_ERR_MISALIGNED;
    return TK_OK;
}

// Whether the two launches around a table (a row per 1024 pairs) beat the three: every workgroup reads the whole table, groups^2 *
// experts words in all.  us on MI355X, three launches / table: 172160 pairs of 32 experts (0.9 Mi words) 15.5 / 8.5, 73728 of 256
// (1.3 Mi) 23.0 / 10.2, 1048576 of 64 (64 Mi) 64 / 30, 2080000 of 32 (128 Mi) 71 / 50, 720000 of 256 (128 Mi) 130 / 44, 524288 of 512
// (128 Mi) 172 / 43; beyond that not measured.  With very few experts the columns are long: one expert, 524288 pairs (512 groups) 26 / 12,
// 2000000 (1954) 40.4 / 41.8, 4000000 60 / 82; two, 4800000 (4688) 77 / 70, 6400000 (6250) 95 / 97, 8000000 112 / 119;
// four, 5600000 (5469) 80 / 76.
static bool table_mapping_pays(int64_t groups, int64_t num_experts) {
    return num_experts <= kSingleMaxExperts && groups <= (1 << 13) && groups * groups * num_experts <= (1 << 27) && groups <= 1800 * (2 * num_experts - 1);
}

// `ws` holds at least tk_fused_mapping_workspace_bytes() bytes
static int launch_fused_mapping(const int64_t *topk_idx, int64_t num_tokens, int num_topk, int num_experts, int alignment,
                                int64_t num_expanded, int32_t *pos_to_expert, int32_t *pos_to_token, int32_t *pos_to_token_topk,
                                int32_t *token_topk_to_pos, int32_t *expert_start, int32_t *expert_end,
                                int32_t *num_tokens_per_expert, int32_t *ws, hipStream_t s, int32_t *host_counts = nullptr) {
    const int numel = (int)(num_tokens * num_topk);
    const int slices = (numel + kSliceElems - 1) / kSliceElems;
    const int blocks = (slices + kWaves - 1) / kWaves;
    const size_t lds = (size_t)kWaves * num_experts * sizeof(int32_t);
    int bits = 0;
    while ((1 << bits) < num_experts) ++bits;
    if (numel > 0 && numel <= kSingleLaunchPairs && num_experts <= kSingleMaxExperts) {
        // A workgroup per 1024 pairs, and no fewer than one per 1024 positions (up to 64): short lists of many experts have far more positions
        // than pairs, and a workgroup beyond the list's end only marks its share of them (us, without / with: 513 pairs of 256 experts, 33024
        // positions 9.8 / 4.6, 4000 pairs, 36480 positions 6.5 / 5.3, 4096 of 512 experts 8.3 / 5.8, 198 of 72, 4672 positions 4.5 / 3.9).
        const int list_groups = (numel + kSingleWaves * kSingleSlice - 1) / (kSingleWaves * kSingleSlice);
        const int groups = std::max(list_groups, (int)std::min<int64_t>(64, (num_expanded + 1023) / 1024));
        hipLaunchKernelGGL(fused_mapping_single_kernel<false>, dim3(groups), dim3(64 * kSingleWaves),
                           (size_t)(1 + kSingleWaves) * num_experts * sizeof(int32_t), s, topk_idx, numel, num_topk, num_experts, bits,
                           alignment, pos_to_expert, pos_to_token, pos_to_token_topk, token_topk_to_pos, expert_start, expert_end,
                           num_tokens_per_expert, (int)num_expanded, nullptr, host_counts);
        return (int)hipGetLastError();
    }
    const int groups = (numel + 1023) / 1024;
    if (numel > 0 && table_mapping_pays(groups, num_experts)) {
        hipLaunchKernelGGL(fused_mapping_table_kernel, dim3(groups), dim3(kThreads), (size_t)num_experts * sizeof(int32_t), s, topk_idx, numel,
                           num_experts, ws);
        hipLaunchKernelGGL(fused_mapping_single_kernel<true>, dim3(groups), dim3(64 * kSingleWaves),
                           (size_t)(2 + kSingleWaves) * num_experts * sizeof(int32_t), s, topk_idx, numel, num_topk, num_experts, bits,
                           alignment, pos_to_expert, pos_to_token, pos_to_token_topk, token_topk_to_pos, expert_start, expert_end,
                           num_tokens_per_expert, (int)num_expanded, ws, host_counts);
        return (int)hipGetLastError();
    }
    // the count launch also fills the padding markers, so it runs even when there are no tokens
    const int fill_blocks = (int)((num_expanded + kThreads - 1) / kThreads);
    const int count_grid = blocks > 0 ? blocks : (fill_blocks > 1024 ? 1024 : fill_blocks);
    if (count_grid > 0)
        hipLaunchKernelGGL(fused_mapping_count_kernel, dim3(count_grid), dim3(kThreads), lds, s, topk_idx, numel, num_experts, ws,
                           pos_to_expert, pos_to_token, pos_to_token_topk, (int)num_expanded);
    hipLaunchKernelGGL(fused_mapping_scan_kernel, dim3(1), dim3(1024), 0, s, ws, slices, num_experts, alignment, expert_start,
                       expert_end, num_tokens_per_expert, host_counts);
    if (blocks > 0)
        hipLaunchKernelGGL(fused_mapping_assign_kernel, dim3(blocks), dim3(kThreads), lds, s, topk_idx, numel, num_topk, num_experts,
                           bits, ws, expert_start, pos_to_expert, pos_to_token, pos_to_token_topk, token_topk_to_pos,
                           (int)num_expanded);
    return (int)hipGetLastError();
}

extern "C" int tk_get_fused_mapping(const int64_t *topk_idx, int64_t num_tokens, int num_topk, int num_experts, int alignment,
                                    int64_t num_expanded, int32_t *pos_to_expert, int32_t *pos_to_token,
                                    int32_t *pos_to_token_topk, int32_t *token_topk_to_pos, int32_t *expert_start,
                                    int32_t *expert_end, int32_t *num_tokens_per_expert, void *workspace,
                                    int64_t workspace_bytes, void *stream) {
    const int rc = tk_check_get_fused_mapping(topk_idx, num_tokens, num_topk, num_experts, alignment, num_expanded, pos_to_expert,
                                              pos_to_token, pos_to_token_topk, token_topk_to_pos, expert_start, expert_end,
                                              num_tokens_per_expert, workspace, workspace_bytes);
    if (rc != TK_OK) return rc;
    return launch_fused_mapping(topk_idx, num_tokens, num_topk, num_experts, alignment, num_expanded, pos_to_expert, pos_to_token,
                                pos_to_token_topk, token_topk_to_pos, expert_start, expert_end, num_tokens_per_expert,
                                static_cast<int32_t *>(workspace), static_cast<hipStream_t>(stream));
}

// The mapping for a caller that needs the segment lengths on the host.  The workgroup that has counted writes them to host memory by itself,
// which saves a copy of num_tokens_per_expert behind the kernels, and the call returns when the stream is through: its caller may go on
// with the lists on any stream, as behind a copy to the host.  us per call of get_fused_mapping on MI355X, copy and wait / this: 329 tokens, top-8,
// 32 experts 26.6 / 20.7; 21520 tokens 32.7 / 27.2.  (Reading on until the words are there and returning then, while positions are still being
// handed out, takes 13.8 and 18.8, and the lists are then in order on this stream only; a loop over hipStreamQuery 32.2 and 39.1.)
extern "C" int tk_get_fused_mapping_with_counts(const int64_t *topk_idx, int64_t num_tokens, int num_topk, int num_experts, int alignment,
                                                int64_t num_expanded, int32_t *pos_to_expert, int32_t *pos_to_token,
                                                int32_t *pos_to_token_topk, int32_t *token_topk_to_pos, int32_t *expert_start,
                                                int32_t *expert_end, int32_t *num_tokens_per_expert, void *workspace,
                                                int64_t workspace_bytes, int32_t *host_counts, void *stream) {
    int rc = tk_check_get_fused_mapping(topk_idx, num_tokens, num_topk, num_experts, alignment, num_expanded, pos_to_expert,
                                        pos_to_token, pos_to_token_topk, token_topk_to_pos, expert_start, expert_end,
                                        num_tokens_per_expert, workspace, workspace_bytes);
    if (rc != TK_OK) return rc;
    if (!host_counts) return TK_ERR_NULL_POINTER;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(s, &capture);
    if (e != hipSuccess) return (int)e;
    if (capture != hipStreamCaptureStatusNone) return TK_ERR_BAD_MODE;      // nothing runs before the capture ends
    void *device = nullptr;
    if (hipHostGetDevicePointer(&device, host_counts, 0) != hipSuccess) {
        (void)hipGetLastError();
        return TK_ERR_BAD_VALUE;
    }
    rc = launch_fused_mapping(topk_idx, num_tokens, num_topk, num_experts, alignment, num_expanded, pos_to_expert, pos_to_token,
                              pos_to_token_topk, token_topk_to_pos, expert_start, expert_end, num_tokens_per_expert,
                              static_cast<int32_t *>(workspace), s, static_cast<int32_t *>(device));
    e = hipStreamSynchronize(s);      // (also where a launch failed: what was launched all the same may still write to host_counts)
    return rc != TK_OK ? rc : (int)e;
}

// ------------------------------------------------------------------------------------------------
// The same mapping for callers that cannot allocate or pass a workspace: the slice x expert table lives in a
// device array owned by the library.  Every GPU holds its own copy of the array at its own address, which is
// looked up once per device (the array's name is only a host-side handle, never a device address) and passed
// to the kernels like the caller's workspace above.  The count launch writes every table entry the later
// launches read, so nothing has to be cleared between calls; calls that overlap on one GPU would share the
// table and race.
static __device__ __align__(256) unsigned char scratch[TK_FUSED_MAPPING_STATIC_BYTES];

// device address of `scratch` on the current device
static int static_scratch_address(void **out) {
    constexpr int kMaxDevices = 64;
    static std::atomic<void *> known[kMaxDevices];
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= kMaxDevices) return TK_ERR_TOO_LARGE;
    void *ptr = known[dev].load(std::memory_order_acquire);
    if (!ptr) {
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return (int)e;
        if (!ptr) return TK_ERR_NULL_POINTER;
        known[dev].store(ptr, std::memory_order_release);
    }
    *out = ptr;
    return TK_OK;
}

extern "C" int tk_get_fused_mapping_static(const int64_t *topk_idx, int64_t num_tokens, int num_topk, int num_experts,
                                           int alignment, int64_t num_expanded, int32_t *pos_to_expert, int32_t *pos_to_token,
                                           int32_t *pos_to_token_topk, int32_t *token_topk_to_pos, int32_t *expert_start,
                                           int32_t *expert_end, int32_t *num_tokens_per_expert, void *stream) {
    // sizes first, so that an oversized request is reported as such whatever else is wrong with it
    if (num_tokens >= 0 && num_topk > 0 && num_experts > 0 && num_experts <= kMaxExperts &&
        num_tokens * num_topk <= INT32_MAX - 1024 &&
        tk_fused_mapping_workspace_bytes(num_tokens, num_topk, num_experts) > (int64_t)TK_FUSED_MAPPING_STATIC_BYTES)
        return TK_ERR_TOO_LARGE;
    void *ws = nullptr;
    int rc = static_scratch_address(&ws);
    if (rc != TK_OK) return rc;
    rc = tk_check_get_fused_mapping(topk_idx, num_tokens, num_topk, num_experts, alignment, num_expanded, pos_to_expert,
                                    pos_to_token, pos_to_token_topk, token_topk_to_pos, expert_start, expert_end,
                                    num_tokens_per_expert, ws, (int64_t)TK_FUSED_MAPPING_STATIC_BYTES);
    if (rc != TK_OK) return rc;
    return launch_fused_mapping(topk_idx, num_tokens, num_topk, num_experts, alignment, num_expanded, pos_to_expert, pos_to_token,
                                pos_to_token_topk, token_topk_to_pos, expert_start, expert_end, num_tokens_per_expert,
                                static_cast<int32_t *>(ws), static_cast<hipStream_t>(stream));
}

extern "C" int tk_check_expand_to_fused(const void *x, int64_t num_tokens, int64_t row_bytes, const int32_t *token_topk_to_pos,
                                        int num_topk, const int32_t *pos_to_expert, int64_t num_expanded, const void *out,
                                        const void *x_sf, int sf_cols, const void *out_sf, int64_t out_sf_ld,
                                        int sf_col_major) {
    if (num_tokens < 0 || num_expanded < 0 || row_bytes <= 0 || num_topk <= 0) return TK_ERR_BAD_SHAPE;
    if (row_bytes % 16 != 0) return TK_ERR_MISALIGNED;
    if (num_tokens + num_expanded > INT32_MAX - 1024) return TK_ERR_TOO_LARGE;
    {   // one workgroup per (token, position, 4 KB chunk) and one per expanded row
        const int64_t chunks = (row_bytes + kExpandChunk - 1) / kExpandChunk;
        if (chunks > INT32_MAX / 8 || num_topk > INT32_MAX / 8) return TK_ERR_TOO_LARGE;
        if (((num_tokens + 7) / 8 * 8) > (INT32_MAX - 1024 - num_expanded) / (num_topk * chunks)) return TK_ERR_TOO_LARGE;
    }
    if (num_expanded > 0 && (!pos_to_expert || !out)) return TK_ERR_NULL_POINTER;
    if (num_tokens > 0 && (!x || !token_topk_to_pos)) return TK_ERR_NULL_POINTER;
    if (!aligned_to(x, 16) || !aligned_to(out, 16)) return TK_ERR_MISALIGNED;
    if (x_sf) {
        if (sf_cols <= 0) return TK_ERR_BAD_SHAPE;
        if (!out_sf) return TK_ERR_NULL_POINTER;
        if (!aligned_to(x_sf, 4) || !aligned_to(out_sf, 4)) return TK_ERR_MISALIGNED;
        if (out_sf_ld < (sf_col_major ? num_expanded : sf_cols)) return TK_ERR_BAD_STRIDE;
    }
    return TK_OK;
}

extern "C" int tk_expand_to_fused(const void *x, int64_t num_tokens, int64_t row_bytes, const int32_t *token_topk_to_pos,
                                  int num_topk, const int32_t *pos_to_expert, int64_t num_expanded, void *out, const void *x_sf,
                                  int sf_cols, void *out_sf, int64_t out_sf_ld, int sf_col_major, void *stream) {
    const int rc = tk_check_expand_to_fused(x, num_tokens, row_bytes, token_topk_to_pos, num_topk, pos_to_expert, num_expanded, out,
                                            x_sf, sf_cols, out_sf, out_sf_ld, sf_col_major);
    if (rc != TK_OK) return rc;
    const int64_t chunks = (row_bytes + kExpandChunk - 1) / kExpandChunk;
    // A workgroup per list entry only for long outputs with many positions per token (see the kernel's comment) and for so few tokens
    // that a workgroup each leaves most compute units without work (full lists of codes with scales, us, EVERY / per token: 32 tokens of
    // 4096 2.9 / 3.2, 64 of 2048, two to a workgroup, 2.75 / 3.0; 64 of 4096 3.1 / 3.3, but 3.2 / 3.05 with one entry of eight live).
    // num_expanded bounds the live entries; a buffer sized for the worst case looks like a full list here.
    const bool many = num_expanded >= 4 * num_tokens;
    // rows of at most half a chunk: several positions of a token, or several tokens, per workgroup
    const int tpr = (int)((row_bytes + 15) / 16);
    const bool short_rows = tpr * 2 <= kThreads;
    const int64_t token_groups = (num_tokens + 7) / 8 * 8;
    const int64_t token_blocks = short_rows ? (num_tokens + kThreads / tpr - 1) / (kThreads / tpr) : token_groups * chunks;
    const bool every = many && (num_expanded * row_bytes >= (int64_t)160 << 20 || token_blocks < 64);
    const int kpw = !short_rows ? 1 : (every && kThreads / tpr > num_topk ? num_topk : kThreads / tpr);
    const int64_t copy_blocks = !every ? token_blocks : token_groups * (short_rows ? (num_topk + kpw - 1) / kpw : num_topk * chunks);
    // padding workgroups take 8 KB of consecutive rows each, two stores per thread.  Measured (us per call, 1 / 2 / 4
    // rows per workgroup): 8 KB rows 64.4 / 69.7 / 71.0; 4 KB rows with scales 41.4 / 36.0 / 37.0
    int pad_rows = row_bytes >= 8192 ? 1 : (int)(8192 / row_bytes > 8 ? 8 : 8192 / row_bytes);
    // Most rows of a long buffer are live where tokens have few positions and it is not much longer than the list: four times the rows per
    // padding workgroup (us, 1 / 2 / 4 times: codes -> [24064, 7168] of 8 ranks 61.5 / 58.9 / 57.7, bf16 -> [33408, 4096], top-2, 76.7 / 72.3 /
    // 70.8; with a third of rows of 2048 padding 18.3 / 17.6 / 17.7; below 16384 rows nothing is won).  With a quarter of the rows certainly
    // padding that many zeros in one place cost more (1 / 4 times: top-2 of bf16 [5000, 7168] -> [16384] 46.2 / 48.6, codes of 4096 14.0 / 16.1; a
    // worst-case buffer of one of 8 ranks, bf16 [8192, 2560] -> [24448], 26.5 / 30.1).
    if (!many && !every && num_expanded >= 16384 && num_expanded * 3 < num_tokens * num_topk * 4) pad_rows *= 4;
    const int64_t grid = copy_blocks + (num_expanded + pad_rows - 1) / pad_rows;
    if (grid == 0) return TK_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
#define TK_EXPAND_LAUNCH(KERNEL, ...)                                                                                       \
    hipLaunchKernelGGL(KERNEL, dim3((unsigned)grid), dim3(kThreads), 0, s, static_cast<const uint8_t *>(x), row_bytes,      \
                       token_topk_to_pos, num_topk, __VA_ARGS__, (int)copy_blocks, (int)num_tokens, (int)num_expanded,      \
                       static_cast<uint8_t *>(out), pos_to_expert, static_cast<const uint32_t *>(x_sf), sf_cols,            \
                       static_cast<uint32_t *>(out_sf), out_sf_ld, sf_col_major, pad_rows)
    if (short_rows) {
        if (every) TK_EXPAND_LAUNCH((expand_short_rows_kernel<true, true>), kpw, tpr);
        else if (x_sf) TK_EXPAND_LAUNCH((expand_short_rows_kernel<false, true>), kpw, tpr);
        else TK_EXPAND_LAUNCH((expand_short_rows_kernel<false, false>), kpw, tpr);
    } else {
        if (every) TK_EXPAND_LAUNCH((expand_to_fused_kernel<true, true>), (int)chunks);
        else if (x_sf) TK_EXPAND_LAUNCH((expand_to_fused_kernel<false, true>), (int)chunks);
        else TK_EXPAND_LAUNCH((expand_to_fused_kernel<false, false>), (int)chunks);
    }
#undef TK_EXPAND_LAUNCH
    return (int)hipGetLastError();
}

extern "C" int tk_check_reduce_fused(const void *x, int x_dtype, int64_t num_expanded, int64_t hidden, const float *x_sf,
                                     const float *topk_weights, const int32_t *token_topk_to_pos, int64_t num_tokens, int num_topk,
                                     const void *out, int out_dtype, const float *sf) {
    (void)x_sf;
    (void)topk_weights;
    (void)sf;
    if (x_dtype != TK_BF16 && x_dtype != TK_F32) return TK_ERR_BAD_DTYPE;
    if (out_dtype != x_dtype && out_dtype != TK_OUT_E4M3) return TK_ERR_BAD_DTYPE;      // same type as the input, or FP8
    if (num_tokens < 0 || num_expanded < 0 || num_topk <= 0 || hidden <= 0 || hidden % 8 != 0) return TK_ERR_BAD_SHAPE;
    if (num_tokens > 65535LL * 65535 || num_expanded > INT32_MAX - 1 || hidden > INT32_MAX - 4096) return TK_ERR_TOO_LARGE;
    if (num_tokens == 0) return TK_OK;
    if (!token_topk_to_pos || !out) return TK_ERR_NULL_POINTER;
    if (num_expanded > 0 && !x) return TK_ERR_NULL_POINTER;
    if (!aligned_to(x, 16) || !aligned_to(out, out_dtype == TK_OUT_E4M3 ? 8 : 16)) return TK_ERR_MISALIGNED;
    if (x_dtype == TK_F32 && !aligned_to(x, 16)) return TK_ERR_MISALIGNED;
    return TK_OK;
}

extern "C" int tk_reduce_fused(const void *x, int x_dtype, int64_t num_expanded, int64_t hidden, const float *x_sf,
                               const float *topk_weights, const int32_t *token_topk_to_pos, int64_t num_tokens, int num_topk,
                               void *out, int out_dtype, const float *sf, void *stream) {
    const int rc = tk_check_reduce_fused(x, x_dtype, num_expanded, hidden, x_sf, topk_weights, token_topk_to_pos, num_tokens,
                                         num_topk, out, out_dtype, sf);
    if (rc != TK_OK || num_tokens == 0) return rc;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (num_expanded == 0) {
        const int64_t words = num_tokens * hidden * (out_dtype == TK_F32 ? 4 : (out_dtype == TK_BF16 ? 2 : 1)) / 8;   // hidden % 8 == 0
        const int64_t blocks = (words + kThreads - 1) / kThreads;
        hipLaunchKernelGGL(reduce_zero_kernel, dim3((unsigned)(blocks < 65536 ? blocks : 65536)), dim3(kThreads), 0, s,
                           static_cast<uint64_t *>(out), words);
        return (int)hipGetLastError();
    }
    const int strips = (int)((hidden + kStripCols - 1) / kStripCols);
    // Pieces side by side in a workgroup: whole rows of up to four, otherwise the largest number up to four that divides the row (five
    // or seven waves 31.5 and 43.5 us instead of 31.0 and 42.8 for bf16 [4096, 2560] and [.., 3584], 8 of 8).  Large launches take two instead
    // of four with more than four terms (bf16 [4096, 4096], 8 of 8: 51.5 / 49.2 us), larger ones with three or four (bf16 [16384, 4096], 3 of 3:
    // 86.8 / 80.9, [8192, 8192] 84.8 / 80.8, but [4500, 8192] 47.8 / 54.9, 4 of 4 58.2 / 56.0; with two terms [32768, 2048] 61.5 / 63.5)
    // and, fp32, one ([8192, 2048], 8 of 8: 102.9 / 99.9; but not rows of a multiple of 16 KB, where some lists lose more than others win:
    // [4500, 4096], 8 of 8, 114.3 / 108.4, [2200, 4096], 7 of 7, 50.8 / 56.0, [8192, 4096], 7 terms of one of 4 ranks, 59.8 / 66.4).
    const int64_t waves = num_tokens * strips;
    const bool bf16 = x_dtype == TK_BF16, few = num_topk <= 2;
    int side = 4;
    while (strips % side) --side;
    if (side == 4 && !few && (num_topk > 4 ? waves > 8192 && (bf16 || hidden % 4096 != 0) : bf16 && waves >= (num_topk == 4 ? 65536 : 98304))) side = bf16 ? 2 : 1;
    // Four waves to a workgroup all the same, on further tokens, since workgroups of one wave are not started fast enough: with one or two
    // terms (bf16 [262144, 256], one term: 69.1 / 61.9 us; fp32 104.3 / 102.9, but [262144, 512] 180 / 186), and with more where there is one
    // piece side by side and the launch is not all latency (one of 8 ranks, 8 terms: bf16 [8192, 2560] 20.7 / 14.8, [8192, 3584] 27.8 / 20.6,
    // [512, 2560] 3.4 / 2.9, 8 of 8 the same within 2 %; but 8 of 8 of fp32 [512, 256] 2.8 / 3.3, [64, 2560] 2.9 / 3.5).
    const bool stacked = few ? (bf16 ? side <= 2 : hidden <= 256) : side == 1 && waves > 2048;
    // HIP takes fewer than 2^32 threads along a grid dimension, and the row tiles of a single column of pieces all ride on x:
    // at most 2^23 row tiles (2^31 threads) per launch.
    const int64_t rows = stacked ? 4 / side : 1, step = rows << 23, out_bytes = out_dtype == TK_F32 ? 4 : (out_dtype == TK_BF16 ? 2 : 1);
    const int cols = strips / side;
    const dim3 block((unsigned)(64 * side * rows));
    for (int64_t t0 = 0; t0 < num_tokens; t0 += step) {
        const int64_t tokens = std::min(num_tokens - t0, step);
        const dim3 grid = tile_grid(cols, (int)((tokens + rows - 1) / rows));
        const int32_t *pos = token_topk_to_pos + t0 * num_topk;
        const float *weights = topk_weights ? topk_weights + t0 * num_topk : nullptr;
        void *o = static_cast<uint8_t *>(out) + t0 * hidden * out_bytes;
#define TK_REDUCE_LAUNCH(T, O)                                                                                              \
    do {                                                                                                                    \
        if (stacked && few) TK_REDUCE_LAUNCH_2(T, O, true, true);                                                           \
        else TK_REDUCE_LAUNCH_MANY(T, O);                                                                                   \
    } while (0)
#define TK_REDUCE_LAUNCH_MANY(T, O)                                                                                         \
    do {                                                                                                                    \
        if (stacked) TK_REDUCE_LAUNCH_2(T, O, true, false);                                                                 \
        else TK_REDUCE_LAUNCH_2(T, O, false, false);                                                                        \
    } while (0)
#define TK_REDUCE_LAUNCH_2(T, O, S, F)                                                                                      \
    hipLaunchKernelGGL((reduce_fused_kernel<T, O, S, F>), grid, block, 0, s, static_cast<const ReduceIn<T>::elem *>(x), pos, \
                       (int)tokens, num_topk, (int)hidden, (int)num_expanded, side | (int)(cols == 1) << 3, weights, x_sf, sf, o)
        if (x_dtype == TK_BF16) {
            if (out_dtype == TK_OUT_E4M3) TK_REDUCE_LAUNCH(bf16_t, 2);
            else TK_REDUCE_LAUNCH(bf16_t, 0);
        } else if (hidden % 512 == 0) {
            if (out_dtype == TK_OUT_E4M3) TK_REDUCE_LAUNCH_MANY(SplitF32, 2);      // (with one or two terms never stacked: rows of 512 and more)
            else TK_REDUCE_LAUNCH_MANY(SplitF32, 1);
        } else {
            if (out_dtype == TK_OUT_E4M3) TK_REDUCE_LAUNCH(float, 2);
            else TK_REDUCE_LAUNCH(float, 1);
        }
#undef TK_REDUCE_LAUNCH_2
#undef TK_REDUCE_LAUNCH_MANY
#undef TK_REDUCE_LAUNCH
    }
    return (int)hipGetLastError();
}
