// Expert grouping for MUL_MAT_ID and the weighted combine of the MoE feed-forward.
#include <algorithm>

#include "actquant_device.h"
#include "qproj_device.h"
#include "qproj_internal.h"

namespace qproj {

// Counting sort of (token, slot) pairs by expert id, one workgroup.  offsets[e]..offsets[e+1]
// indexes the pairs of expert e inside order[]; active[] is the work list (active_slots_offset): the experts that
// have pairs, or tiles of them (those with more than heavy_above pairs first: launch_moe_group, ascending within both parts).
// Ids outside [0, n_expert) raise *error_flag and their pairs are left out (their outputs are not written).  Offsets and work
// list follow from the counts alone, so repeated runs produce the same launch geometry; the order of an expert's pairs inside
// order[] does not (moe_group_kernel below), and nothing that reads order[] may depend on it.
//
// Two ways to sort.  Up to 1536 experts a counter a wave and expert in LDS (moe_group_kernel).  Beyond, sweeps: each of
// the 16 waves takes every 16th expert and sweeps the pair list 64 ids at a time (consecutive lanes on consecutive ids);
// a ballot of the matches gives the count in the first sweep and, with the number of matching lanes below one's own, the slot
// in the second: ascending pair order.  (A version that read the ids from LDS inside the sweeps was a chain of dependent loads:
// 19 us for 512 pairs and 128 experts.)
constexpr int kGroupThreads = 1024;
constexpr int kGroupLdsIds = 8192;   // pair ids staged in LDS up to this many, read from global beyond

// inclusive prefix sum over the wave, in the vector unit: within a row of 16 lanes, then rows onto the next ones
__device__ __forceinline__ int wave_prefix(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
    return v;
}
// sum over the 16 lanes of a row, in every lane
__device__ __forceinline__ int row_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, true);   // row_ror:8, 4, 2, 1
    v += __builtin_amdgcn_update_dpp(0, v, 0x124, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x122, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x121, 0xf, 0xf, true);
    return v;
}

// cnt[e] = pairs of expert e on entry; on exit cnt[e] = offsets[e] = its first slot, active[] lists the
// experts that have pairs.  All threads of the workgroup call it; the caller synchronizes afterwards.
// PER: experts a thread (1 up to 1024 experts, 8 beyond).  The launch waits for this one workgroup: with the scans through LDS
// shuffles, eight experts a thread whatever their number and the tiles of an expert by a division it was four of the seven
// microseconds of the grouping launch.
template <int PER>
__device__ __forceinline__ void group_scan_per(int n_expert, int32_t *cnt, int32_t *wsum, int32_t *__restrict__ offsets,
                                               int32_t *__restrict__ active, int heavy_above, bool tiled, int list_cap) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // exclusive scans over the workgroup (in the vector unit inside a wave, wave totals through LDS) of the pair
    // counts (-> offsets) and of the non-empty flags (-> compact list of the experts that have work);
    // thread t owns experts [t * PER, t * PER + PER)
    int tot[PER], local = 0, local_f = 0, local_h = 0;
    // list positions of an expert: one, or one per tile of its pairs
    static_assert(kMoeTileRows == 64, "tiles of an expert's pairs by a shift");
    auto positions = [&](int pairs) { return tiled ? (pairs + 63) >> 6 : (int)(pairs > 0); };
    // The experts with more pairs than one pass of the grouped kernels stages (two passes over their weights) go
    // to the front of the list, everything else stays in ascending order: the grouped kernels hand their
    // workgroups out in list order, and a two-pass expert then starts with the grid instead of stretching its
    // tail.  A third scan, over the "heavy" flags, gives the positions.  (The whole list ordered by pair count
    // evened the launches out as well but cost the ordinary case 3 us: neighbouring workgroups no longer read
    // neighbouring experts.)
    auto is_heavy = [&](int pairs) { return heavy_above > 0 && pairs > heavy_above; };
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = tid * PER + i;
        tot[i] = e < n_expert ? cnt[e] : 0;
        local += tot[i];
        local_f += positions(tot[i]);
        local_h += is_heavy(tot[i]) ? positions(tot[i]) : 0;
    }
    const int incl = wave_prefix(local), incl_f = wave_prefix(local_f), incl_h = wave_prefix(local_h);
    if (lane == 63) {
        wsum[wave] = incl;
        wsum[16 + wave] = incl_f;
        wsum[32 + wave] = incl_h;
    }
    __syncthreads();
    // what the waves before this one counted: a wave total a lane of each row
    static_assert(kGroupThreads / 64 == 16, "a row of lanes holds the totals of the waves");
    const int w = lane & 15, w0 = wsum[w], w1 = wsum[16 + w], w2 = wsum[32 + w];
    int before = incl - local + row_sum(w < wave ? w0 : 0), before_f = incl_f - local_f + row_sum(w < wave ? w1 : 0),
        before_h = incl_h - local_h + row_sum(w < wave ? w2 : 0);
    const int n_heavy = row_sum(w2);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = tid * PER + i;
        if (e < n_expert) {
            cnt[e] = before;   // from here on: the expert's first slot
            offsets[e] = before;
            before += tot[i];
            if (tot[i] > 0) {
                const bool heavy = is_heavy(tot[i]);
                const int pos = heavy ? before_h : n_heavy + (before_f - before_h);
                int4 *rec = reinterpret_cast<int4 *>(active + active_slots_offset(list_cap)) + pos;
                const int n_pos = positions(tot[i]);
                if (tiled) {
                    for (int t = 0; t < n_pos; ++t) rec[t] = make_int4(e, before - tot[i] + t * 64, min(64, tot[i] - t * 64), 0);
                } else {
                    active[pos] = e;
                    *rec = make_int4(e, before - tot[i], tot[i], 0);
                }
                before_f += n_pos;
                before_h += heavy ? n_pos : 0;
            }
        }
    }
    if (tid == kGroupThreads - 1) {
        offsets[n_expert] = before;
        active[list_cap] = before_f;   // positions of the list
    }
}
__device__ __forceinline__ void group_scan(int n_expert, int32_t *cnt, int32_t *wsum, int32_t *__restrict__ offsets,
                                           int32_t *__restrict__ active, int heavy_above, bool tiled, int list_cap) {
    if (n_expert <= kGroupThreads) group_scan_per<1>(n_expert, cnt, wsum, offsets, active, heavy_above, tiled, list_cap);
    else group_scan_per<8>(n_expert, cnt, wsum, offsets, active, heavy_above, tiled, list_cap);
}

template <bool STAGED>
__device__ __forceinline__ void group_sweeps(const int32_t *__restrict__ ids, const int32_t *sid, int n_pairs, int n_expert,
                                             int32_t *cnt, int32_t *wsum, int32_t *__restrict__ order,
                                             int32_t *__restrict__ offsets, int32_t *__restrict__ active, int heavy_above,
                                             bool tiled, int list_cap) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    constexpr int kWaves = kGroupThreads / 64;
    auto id_at = [&](int p) { return p < n_pairs ? (STAGED ? sid[p] : ids[p]) : -1; };
    // A lane keeps the ids of its positions in registers, kHeld at a time (1024 pairs per wave and block),
    // and runs through its experts on them: the sweeps are ballots on registers, not a chain of loads.
    constexpr int kHeld = 16;
    // sweep 1: pairs per expert (cnt starts at zero)
    for (int base = 0; base < n_pairs; base += 64 * kHeld) {
        int v[kHeld];
#pragma unroll
        for (int u = 0; u < kHeld; ++u) v[u] = id_at(base + 64 * u + lane);
        for (int e = wave; e < n_expert; e += kWaves) {
            int c = 0;
#pragma unroll
            for (int u = 0; u < kHeld; ++u) c += __popcll(__ballot(v[u] == e));
            if (lane == 0) cnt[e] += c;   // every expert belongs to one wave
        }
    }
    __syncthreads();
    group_scan(n_expert, cnt, wsum, offsets, active, heavy_above, tiled, list_cap);
    __syncthreads();
    // sweep 2: placement, ascending pair order inside every expert (cnt[e] = the expert's next free slot)
    for (int base = 0; base < n_pairs; base += 64 * kHeld) {
        int v[kHeld];
#pragma unroll
        for (int u = 0; u < kHeld; ++u) v[u] = id_at(base + 64 * u + lane);
        for (int e = wave; e < n_expert; e += kWaves) {
            int w = cnt[e];
#pragma unroll
            for (int u = 0; u < kHeld; ++u) {
                const bool mine = v[u] == e;
                const unsigned long long m = __ballot(mine);
                if (mine)
                    order[w + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0))] =
                        base + 64 * u + lane;
                w += __popcll(m);
            }
            if (lane == 0) cnt[e] = w;
        }
    }
}

// The sweeps above cost n_expert x n_pairs / 1024 steps.  While a table of 16 counters an expert fits LDS the work is made
// proportional to n_pairs instead: a wave takes a contiguous sixteenth of the pairs and adds one to its own counter of
// each pair's expert (the LDS hands every lane the count before it), a prefix over the 16 waves per expert and the scan over
// the experts follow, and every pair knows its slot: first[expert] + before[wave][expert] + count in the wave.  Pairs of
// an expert ascend from one 64 to the next; inside a 64 their order is the LDS's (no result depends on it).  Pairs beyond
// the blocks whose counts a lane keeps in registers are counted a second time when they are placed.
// (128 experts, traced, quantizer of the token rows in the spare workgroups: ranks from ballots on the bits of the id and a
// counter per 64 pairs and expert 14.7 us at 4000 pairs, and 159 us at 16384, which were left to the sweeps; this 10.1 and
// 19.7; 512 pairs 7.1 either way.)
constexpr int kHeldBlocks = 8;

__global__ __launch_bounds__(kGroupThreads) void moe_group_kernel(const int32_t *__restrict__ ids, int n_pairs,
                                                                  int n_expert, int32_t *__restrict__ order,
                                                                  int32_t *__restrict__ offsets,
                                                                  int32_t *__restrict__ active,
                                                                  int32_t *__restrict__ error_flag, int by_block,
                                                                  int heavy_above, int tiled, int list_cap,
                                                              const RowQuantJob job) {
    // Workgroups past the first have nothing to do with the grouping: they quantize the activation rows the
    // grouped projection is going to read (one 256-wide chunk a wave, ggml's quantize_row_q8_K as in the
    // standalone quantizer), so that the two passes, which depend only on the call's inputs, share a launch.
    if (blockIdx.x > 0) {
        const int64_t sb = (int64_t)(blockIdx.x - 1) * (kGroupThreads / 64) + (threadIdx.x >> 6);
        if (sb < job.n_super) {   // whole wave decides together
            const int lane = threadIdx.x & 63;
            const float4 v = reinterpret_cast<const float4 *>(job.x + sb * 256)[lane];
            wave_store_q8k(v, lane, sb, job.qs, job.d, job.bsums, job.hsum);
        }
        return;
    }
    extern __shared__ int32_t lds[];
    int32_t *cnt = lds;                 // [n_expert] pairs of the expert, then its first slot
    int32_t *wsum = cnt + n_expert;     // [48] wave totals of the three scans
    int32_t *tab = wsum + 48;           // by_block: [16 waves][n_expert]; else the staged ids
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (!by_block) {
        const bool staged = n_pairs <= kGroupLdsIds;
        bool bad = false;
        for (int p = tid; p < n_pairs; p += kGroupThreads) {
            const int e = ids[p];
            bad |= e < 0 || e >= n_expert;
            if (staged) tab[p] = e;
        }
        for (int e = tid; e < n_expert; e += kGroupThreads) cnt[e] = 0;
        if (bad) atomicOr(error_flag, 1);
        __syncthreads();
        if (staged) group_sweeps<true>(ids, tab, n_pairs, n_expert, cnt, wsum, order, offsets, active, heavy_above, tiled, list_cap);
        else group_sweeps<false>(ids, tab, n_pairs, n_expert, cnt, wsum, order, offsets, active, heavy_above, tiled, list_cap);
        return;
    }
    const int n_blocks = (n_pairs + 63) / 64, per_wave = (n_blocks + kGroupThreads / 64 - 1) / (kGroupThreads / 64);
    const int b0 = wave * per_wave, nb = max(0, min(per_wave, n_blocks - b0));   // the wave's blocks
    int32_t *mine = tab + wave * n_expert;
    int vid[kHeldBlocks], slot[kHeldBlocks];
    bool bad = false;
    auto id_at = [&](int b) {
        const int p = 64 * (b0 + b) + lane;
        int v = b < nb && p < n_pairs ? ids[p] : -1;
        bad |= b < nb && p < n_pairs && (v < 0 || v >= n_expert);
        return v >= n_expert ? -1 : v;
    };
#pragma unroll
    for (int i = 0; i < kHeldBlocks; ++i) vid[i] = id_at(i);   // the loads first: they travel while the table is cleared
    for (int t = tid; t < (kGroupThreads / 64) * n_expert; t += kGroupThreads) tab[t] = 0;
    __syncthreads();
    // the pair's place among the wave's pairs of its expert
    auto place = [&](int v) {
        return v >= 0 ? __hip_atomic_fetch_add(&mine[v], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) : 0;
    };
#pragma unroll
    for (int i = 0; i < kHeldBlocks; ++i)
        if (i < nb) slot[i] = place(vid[i]);   // wave-uniform
    for (int b = kHeldBlocks; b < nb; b += 4) {
        int v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = id_at(b + u);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (b + u < nb) place(v[u]);
    }
    if (bad) atomicOr(error_flag, 1);
    __syncthreads();
    // per expert: counts of the waves -> pairs of the waves before; total
    for (int e = tid; e < n_expert; e += kGroupThreads) {
        int c[kGroupThreads / 64], run = 0;
#pragma unroll
        for (int w = 0; w < kGroupThreads / 64; ++w) c[w] = tab[w * n_expert + e];
#pragma unroll
        for (int w = 0; w < kGroupThreads / 64; ++w) {
            tab[w * n_expert + e] = run;
            run += c[w];
        }
        cnt[e] = run;
    }
    __syncthreads();
    group_scan(n_expert, cnt, wsum, offsets, active, heavy_above, tiled, list_cap);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kHeldBlocks; ++i)
        if (i < nb && vid[i] >= 0) order[cnt[vid[i]] + mine[vid[i]] + slot[i]] = 64 * (b0 + i) + lane;
    if (nb <= kHeldBlocks) return;
    // the wave's counters move past the blocks placed so far; the others are ranked again
#pragma unroll
    for (int i = 0; i < kHeldBlocks; ++i) place(vid[i]);
    for (int b = kHeldBlocks; b < nb; b += 4) {
        int v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = id_at(b + u);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (b + u < nb) {
                const int at = place(v[u]);
                if (v[u] >= 0) order[cnt[v[u]] + at] = 64 * (b0 + b + u) + lane;
            }
    }
}

hipError_t launch_moe_group(const int32_t *ids, int64_t n_pairs, int64_t n_expert, int32_t *order,
                            int32_t *offsets, int32_t *active, int32_t *error_flag, int64_t pass_rows,
                            const RowQuantJob *quantize, hipStream_t s, int64_t tile_rows) {
    if (n_expert > 8192 || n_pairs > 0x7fffffff || (tile_rows && tile_rows != kMoeTileRows)) return hipErrorInvalidValue;
    const size_t table = (size_t)(kGroupThreads / 64) * (size_t)n_expert;
    const bool by_block = table <= 24 * 1024;   // at most 96 KB of LDS
    const size_t lds = ((size_t)n_expert + 48 + (by_block ? table : n_pairs <= kGroupLdsIds ? (size_t)n_pairs : 0)) * sizeof(int32_t);
    // Which experts start first: those that need a pass over their weights more than the average one.  `pass_rows`: rows a
    // pass of the grouped kernel behind this stages (mfma_grouped_pass_rows); the line is the multiple of that below the
    // average, or above it from three eighths of a pass on, where nearly every expert would be beyond the one below (at 31 pairs
    // an expert and 32 rows those with more than 32 take two passes; with the line at 16 nothing was ordered there and the
    // launches waited for two-pass experts begun last: 500 tokens, 128 experts, top-8 of 2048 x 768 234 -> 207 us; 16 rows, line
    // below / above the average: 22 pairs 257 / 229, 50 pairs 375 / 406, 19 pairs 299 / 324, 87 pairs 474 / 452).
    // (The same line for a list of tiles: the experts with the most and the fullest tiles.  500 tokens: those with more than 32
    // pairs, two token tiles of the matrix instruction, so that every compute unit gets one such workgroup and one lighter.)
    const int64_t heavy = pass_rows * std::max<int64_t>(1, (n_pairs / n_expert + pass_rows * 5 / 8) / pass_rows);
    const int64_t list_cap = moe_list_capacity(n_expert, n_pairs, tile_rows);
    if (list_cap > 0x7fffffff) return hipErrorInvalidValue;
    if (dry_run()) {
        plan_note("moe_group_kernel: %lld pairs over %lld experts (%s), those with more than %lld first%s", (long long)n_pairs, (long long)n_expert,
                  by_block ? "counters a wave and expert" : "ballot sweeps per expert", (long long)heavy,
                  quantize ? ", spare workgroups quantize the token rows" : "");
        return hipSuccess;
    }
    static LdsLimit limit;
    const hipError_t e = limit.allow(&moe_group_kernel, lds);
    if (e != hipSuccess) return e;
    RowQuantJob job{};
    if (quantize) job = *quantize;
    const int64_t extra = (job.n_super + kGroupThreads / 64 - 1) / (kGroupThreads / 64);
    if (extra >= 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL(moe_group_kernel, dim3((unsigned)(1 + extra)), dim3(kGroupThreads), lds, s, ids, (int)n_pairs,
                       (int)n_expert, order, offsets, active, error_flag, by_block ? 1 : 0,
                       (int)heavy, tile_rows ? 1 : 0, (int)list_cap, job);
    return hipGetLastError();
}

// y[b][c] = e[b][0][c]*w[b][0] + e[b][1][c]*w[b][1] + ... in slot order, each product rounded
// before it is added (llama.cpp multiplies by the routing weights, then adds the expert views
// one after the other).  Bound: HBM, n_used floats read for one written; V columns a thread, eight slots requested
// before the first is used.
template <int V>
__global__ __launch_bounds__(256) void moe_combine_kernel(const float *__restrict__ e, const float *__restrict__ w,
                                                          int64_t n, int n_used, uint32_t N, float *__restrict__ y) {
    typedef float vec __attribute__((ext_vector_type(V)));
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
    if (i >= n) return;
    const int64_t b = n <= 0xffffffffll ? (int64_t)((uint32_t)i / N) : i / N, c = i - b * N;   // V columns of one row
    const float *src = e + b * n_used * N + c, *wt = w + b * n_used;
    vec s = (vec)0.f;
    for (int j0 = 0; j0 < n_used; j0 += 8) {
        vec v[8];
        float f[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (j0 + u < n_used) {
                v[u] = *reinterpret_cast<const vec *>(src + (int64_t)(j0 + u) * N);
                f[u] = wt[j0 + u];
            }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (j0 + u < n_used) {
#pragma unroll
                for (int k = 0; k < V; ++k) {
                    const float p = __fmul_rn(v[u][k], f[u]);
                    s[k] = j0 + u == 0 ? p : __fadd_rn(s[k], p);
                }
            }
    }
    *reinterpret_cast<vec *>(y + i) = s;
}

// h = silu(g) * u with ggml's expression for silu, x / (1 + expf(-x))
__global__ __launch_bounds__(256) void swiglu_kernel(const float *__restrict__ g, const float *__restrict__ u, size_t n,
                                                     float *__restrict__ h) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) {
        const float x = g[i];
        h[i] = (x / (1.0f + expf(-x))) * u[i];
    }
}

hipError_t launch_swiglu(const float *g, const float *u, size_t n, float *h, hipStream_t s) {
    if (n == 0) return hipSuccess;
    if (dry_run()) {
        plan_note("swiglu_kernel: %zu elements", n);
        return hipSuccess;
    }
    hipLaunchKernelGGL(swiglu_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, g, u, n, h);
    return hipGetLastError();
}

hipError_t launch_moe_combine(const float *e, const float *weights, int64_t B, int64_t n_used, int64_t N,
                              float *y, hipStream_t s) {
    const int64_t n = B * N;
    if (n == 0) return hipSuccess;
    if (dry_run()) {
        plan_note("moe_combine_kernel: %lld tokens x %lld, %lld experts a token in slot order", (long long)B, (long long)N, (long long)n_used);
        return hipSuccess;
    }
    if (N > 0xffffffffll || n > 0x7fffffffll * 256) return hipErrorInvalidValue;
    // Four columns a thread where that leaves a workgroup and more a compute unit (one column: 500 / 2048 tokens of 2048
    // columns and 8 experts 9.2 / 41.4 us, four: 7.3 / 23.1; at 64 tokens four lost, 99.2 -> 101.0 a call of the feed-forward).
    const bool wide = N % 4 == 0 && n >= 4 * 256 * 256 && ((reinterpret_cast<uintptr_t>(e) | reinterpret_cast<uintptr_t>(y)) & 15) == 0;
    if (wide) hipLaunchKernelGGL(moe_combine_kernel<4>, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, s, e, weights, n, (int)n_used, (uint32_t)N, y);
    else hipLaunchKernelGGL(moe_combine_kernel<1>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, e, weights, n, (int)n_used, (uint32_t)N, y);
    return hipGetLastError();
}

}  // namespace qproj
