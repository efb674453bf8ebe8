// Expert feed-forward batches on the int8 matrix cores: Q4_K experts x ggml Q8_K activations, up to 64 (token, slot)
// pairs of an expert per pass over its weights.
//
// Bound on paper: HBM over the bytes of the experts a call touches.
//   - The grouping pass lists tiles {expert, first pair, up to 64 pairs}; a workgroup (4 waves, two workgroups a compute
//     unit up to 7936 weights a row) takes one tile and `tiles_n` row tiles of its expert as ONE stream of (row tile, super-block) steps, so the
//     pipeline never restarts: raw weight blocks go straight from global memory into wave-private LDS strips two steps
//     ahead, the gathered activation rows (any row per lane: the loads into LDS take an address each) one step ahead into
//     a buffer that the four waves share, one barrier a step.
//   - A wave owns 32 columns of the matrix instruction.  Gate and up share them (16 rows each), so that gate_r . x and
//     up_r . x of a token end up sixteen lanes apart and silu(gate) * up is formed in registers.
//   - A tile of at most 32 pairs runs the instance with one token tile: half the matrix instructions and flushes.
// Sums are those of the grouped small-batch kernel, bit for bit: the exact integer dot product of a super-block (both
// base-8 digits of the scales as int8 operands, see gemm_q4k_q8k_direct_kernel), the exact integer sum of mins x code
// sums (fp16 operands, fp32 sums of integers below 2^24), one rounding each for d * I, dmin * S, their difference and
// the fma into the running sum, super-blocks in ascending order.
#include <algorithm>

#include "gemm_convert.h"
#include "lds_direct.h"
#include "qproj_device.h"
#include "qproj_internal.h"

namespace qproj {

namespace {

constexpr int kWaves = 4, kThreads = 64 * kWaves;
constexpr int kMaxJT = kMoeTileRows / 32;
constexpr int kStripBytes = 32 * 144, kStripLoads = 5;

struct MoeStreamArgs {
    const uint8_t *w0, *w1;   // blocks of the expert stack; w1: the up projection of the SwiGLU launch
    float *y;                 // [pairs][N]
    const int8_t *qs;         // activation rows, their scales and sums of 16 codes (fp16)
    const float *d;
    const uint16_t *hsum;
    const int32_t *order;     // pairs sorted by expert
    const int4 *tiles;        // {expert, first slot of order[], pairs, -}
    const int32_t *n_tiles;
    int64_t N;
    int nb, x_div;            // activation row of pair p is p / x_div
    int wgs_per_tile, row_tiles;   // workgroups that share a tile; row tiles each of them walks
    int list_capacity;
};

// LDS: activations [2][64 tokens][256] (16-byte segments XOR-swizzled by the token), sums [2][64][16] fp16, strips
// [2][4 waves][32 rows x 144 B], the pair of each token, activation scales [nb][64]
constexpr int kOffSum = 2 * kMaxJT * 8192, kOffStrip = kOffSum + 2 * kMaxJT * 1024,
              kOffPair = kOffStrip + 2 * kWaves * kStripBytes, kOffDx = kOffPair + kMoeTileRows * 4;
constexpr int moe_stream_lds(int nb) { return kOffDx + nb * kMoeTileRows * 4; }
constexpr int workgroups_per_cu(int nb) { return 2 * moe_stream_lds(nb) <= 160 * 1024 ? 2 : 1; }   // (the launch bounds: two at most)

// eight fp16 integers: the four bytes of `w` (below 128), each twice
__device__ __forceinline__ v8h bytes_twice_to_f16(uint32_t w) {
    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
    const v2h k = {(_Float16)1024.f, (_Float16)1024.f};
    v8h r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {   // 0x6400 | b is 1024 + b
        const v2h h = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, w, 0x04000400u | (uint32_t)(i << 16) | (uint32_t)i)) - k;
        r[2 * i] = h[0];
        r[2 * i + 1] = h[1];
    }
    return r;
}

template <bool SWIGLU, int JT>
__device__ __forceinline__ void moe_stream_tile(const MoeStreamArgs &g, uint8_t *smem, const int4 tile, int part) {
    constexpr int TM = 32 * JT, kRows = SWIGLU ? 16 : 32;   // weight rows of a wave's row tile
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, lh = lane >> 5;
    const int nb = g.nb, count = tile.z;
    const int64_t N = g.N;
    const int64_t n_row_tiles = (N + kWaves * kRows - 1) / (kWaves * kRows), rt0 = (int64_t)part * g.row_tiles;
    const int n_rt = (int)min((int64_t)g.row_tiles, n_row_tiles - rt0);
    if (n_rt <= 0) return;   // the whole workgroup

    // ---- weights: piece p of a strip is bytes 16 (p % 9).. of row p / 9.  The 288 pieces are four and a half requests: the fifth
    // asks for the last 64, half of them a second time with the same bytes for the same place, so that a strip ends where its rows
    // end (with 512 spare bytes behind each of the eight, a second workgroup did not fit beside rows of 4096 weights)
    uint8_t *const strip = smem + kOffStrip + wave * kStripBytes;   // second buffer kWaves * kStripBytes further on
    const uint8_t *src[kStripLoads];
    auto strip_row_tile = [&](int rt) {
        const int64_t row0 = ((rt0 + rt) * kWaves + wave) * kRows;
#pragma unroll
        for (int c = 0; c < kStripLoads; ++c) {
            const int p = lane + (c < 4 ? 64 * c : 288 - 64), r = p / 9;
            const int64_t row = min(row0 + (r & (kRows - 1)), N - 1);   // rows past the edge repeat the last (never stored)
            src[c] = (SWIGLU && r >= 16 ? g.w1 : g.w0) + ((int64_t)tile.x * N + row) * nb * 144 + 16 * (p - 9 * r);
        }
    };
    const int n_steps = n_rt * nb;
    int req_rt = 0, req_sb = 0;   // the step that was requested last
    auto request_strip = [&](uint8_t *dst) {
#pragma unroll
        for (int c = 0; c < kStripLoads; ++c) global_to_lds16(src[c], dst + (c < 4 ? 1024 * c : kStripBytes - 1024));
    };
    auto advance = [&]() {   // (past the last step: stays there)
        if (++req_sb < nb) {
#pragma unroll
            for (int c = 0; c < kStripLoads; ++c) src[c] += 144;
        } else if (req_rt + 1 < n_rt) {
            req_sb = 0;
            strip_row_tile(++req_rt);
        }
    };
    strip_row_tile(0);

    // ---- activations: request j of a wave = tokens 4 (wave + 4 j) .. +3; every lane follows its own row.  Loads return in
    // order: the pairs first, then the weights of the first step, and the rows while those are on their way from HBM.
    constexpr int AP = 8 * JT / kWaves;
    auto pair_of = [&](int tok) { return g.order[tile.y + min(tok, count - 1)]; };
    auto token_of = [&](int j) { return 4 * (wave + kWaves * j) + (lane >> 4); };
    int apair[AP];
#pragma unroll
    for (int j = 0; j < AP; ++j) apair[j] = pair_of(token_of(j));
    const int hpair = pair_of((wave % JT) * 32 + (lane >> 1)), tpair = pair_of(tid % TM);
    __builtin_amdgcn_sched_barrier(0);
    request_strip(strip);
    __builtin_amdgcn_sched_barrier(0);
    const int8_t *asrc[AP];
#pragma unroll
    for (int j = 0; j < AP; ++j)
        asrc[j] = g.qs + (int64_t)(apair[j] / g.x_div) * nb * 256 + 16 * ((lane & 15) ^ (token_of(j) & 15));
    const uint16_t *const hsrc = g.hsum + (int64_t)(hpair / g.x_div) * nb * 16 + 8 * (lane & 1);
    auto request_acts = [&](int sb, int buf) {
#pragma unroll
        for (int j = 0; j < AP; ++j) global_to_lds16(asrc[j] + sb * 256, smem + (buf * kMaxJT) * 8192 + (wave + kWaves * j) * 1024);
        if (wave < JT) global_to_lds16(hsrc + sb * 16, smem + kOffSum + (buf * kMaxJT + wave) * 1024);
    };
    request_acts(0, 0);
    advance();
    request_strip(strip + kWaves * kStripBytes);   // (of a single step: once more)
    float *const dx_lds = reinterpret_cast<float *>(smem + kOffDx);
    int *const pair_lds = reinterpret_cast<int *>(smem + kOffPair);
    if (tid < TM) pair_lds[tid] = tpair;
    {
        const float *drow = g.d + (int64_t)(tpair / g.x_div) * nb;
        for (int sb = tid / TM; sb < nb; sb += kThreads / TM) dx_lds[sb * TM + tid % TM] = drow[sb];
    }
    wait_vmcnt<0>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    v16f acc[JT];
    const v16i zi = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const v16f zf = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < JT; ++j) acc[j] = zf;
    const int aoffl = l32 * 256 + 16 * ((8 * lh) ^ (l32 & 15));

    // accumulator register v of lane l is token 8 (v / 4) + 4 (l / 32) + v % 4, column l % 32
    auto store_row_tile = [&](int rt) {
        const int64_t row0 = ((rt0 + rt) * kWaves + wave) * kRows;
        const int64_t n = row0 + (SWIGLU ? lane & 15 : l32);
        const bool up_lane = SWIGLU && (lane & 16);
#pragma unroll
        for (int j = 0; j < JT; ++j) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m0 = j * 32 + 8 * i + 4 * lh;
                const v4i pair = *reinterpret_cast<const v4i *>(pair_lds + m0);
                if constexpr (SWIGLU) {
                    // lanes of the gate finish the even tokens, lanes of the up projection the odd ones
#pragma unroll
                    for (int r = 0; r < 4; r += 2) {
                        const float even = acc[j][4 * i + r], odd = acc[j][4 * i + r + 1];
                        const float got = __shfl_xor(up_lane ? even : odd, 16);
                        const float gate = up_lane ? got : even, up = up_lane ? odd : got;
                        const int m = m0 + r + (up_lane ? 1 : 0);
                        if (m < count && n < N) g.y[(int64_t)(up_lane ? pair[r + 1] : pair[r]) * N + n] = (gate / (1.0f + expf(-gate))) * up;
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (m0 + r < count && n < N) g.y[(int64_t)pair[r] * N + n] = acc[j][4 * i + r];
                }
            }
            acc[j] = zf;
        }
    };

    auto step = [&](int s, int sb, auto more1, auto more2) {
        constexpr bool MORE1 = decltype(more1)::value, MORE2 = decltype(more2)::value;
        uint8_t *const sbuf = strip + (s & 1) * kWaves * kStripBytes;
        v4i q[4];
        const v4i hdr = *reinterpret_cast<const v4i *>(sbuf + l32 * 144);
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = *reinterpret_cast<const v4i *>(sbuf + l32 * 144 + 16 + 64 * lh + 16 * i);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the strip has been read: it may be overwritten
        if constexpr (MORE1) request_acts(sb + 1 == nb ? 0 : sb + 1, (s + 1) & 1);
        if constexpr (MORE2) {
            advance();
            request_strip(sbuf);
        }
        __builtin_amdgcn_sched_barrier(0);   // the requests stay ahead of the arithmetic they overlap with

        const uint8_t *const ab = smem + (s & 1) * kMaxJT * 8192;
        auto frag = [&](int j, int i) { return *reinterpret_cast<const v4i *>(ab + j * 8192 + (aoffl ^ (16 * i))); };
        const ScalesK4 sc = unpack_scales_k4((uint32_t)hdr[1], (uint32_t)hdr[2], (uint32_t)hdr[3]);
        const uint32_t scw = lh ? sc.sc_hi : sc.sc_lo;   // sub-blocks 4 (l / 32) .. +3
        const uint32_t lo_w = scw & 0x07070707u, hi_w = (scw >> 3) & 0x07070707u;
        v4i cl[2], ch[2], af[3][JT];
        v16i ilo[JT], ihi[JT];
        v16f msum[JT];
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int j = 0; j < JT; ++j) af[p][j] = frag(j, p);
        convert_q4k(q[0], lo_w, hi_w, 0, cl[0], ch[0]);
        __builtin_amdgcn_sched_barrier(0);
        v8h mins, am[JT];
#pragma unroll
        for (int p = 0; p < 8; ++p) {
            // the activation fragments of two products are in flight, the next product's weights are converted between
            // the matrix instructions of this one
            if (p + 2 < 8) {
#pragma unroll
                for (int j = 0; j < JT; ++j) af[(p + 2) % 3][j] = frag(j, p + 2);
            }
            if (p + 1 < 8) convert_q4k(q[2 * ((p + 1) >> 2) + ((p + 1) & 1)], lo_w, hi_w, (p + 1) >> 1, cl[(p + 1) & 1], ch[(p + 1) & 1]);
            if (p == 5) {
                mins = bytes_twice_to_f16(lh ? sc.mn_hi : sc.mn_lo);
#pragma unroll
                for (int j = 0; j < JT; ++j) am[j] = *reinterpret_cast<const v8h *>(smem + kOffSum + ((s & 1) * kMaxJT + j) * 1024 + l32 * 32 + 16 * lh);
            }
#pragma unroll
            for (int j = 0; j < JT; ++j) {
                ilo[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[p % 3][j], cl[p & 1], p == 0 ? zi : ilo[j], 0, 0, 0);
                ihi[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[p % 3][j], ch[p & 1], p == 0 ? zi : ihi[j], 0, 0, 0);
            }
            if (p == 7) {
#pragma unroll
                for (int j = 0; j < JT; ++j) msum[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(am[j], mins, zf, 0, 0, 0);
            }
#pragma unroll
            for (int k = 0; k < 2 * JT; ++k) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        const float dw = h2f((uint32_t)hdr[0] & 0xffffu), dmin = h2f((uint32_t)hdr[0] >> 16);
#pragma unroll
        for (int j = 0; j < JT; ++j) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // (as v4i: a float4 read here makes the compiler wait for every outstanding request to LDS first)
                const v4i d4 = *reinterpret_cast<const v4i *>(dx_lds + sb * TM + j * 32 + 8 * i + 4 * lh);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int v = 4 * i + r;
                    const float t = dw * (float)((ihi[j][v] << 3) + ilo[j][v]) - dmin * msum[j][v];
                    acc[j][v] = fmaf(__int_as_float(d4[r]), t, acc[j][v]);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (MORE1) {
            if constexpr (MORE2) wait_vmcnt<kStripLoads>();   // all but the strip just asked for
            else wait_vmcnt<0>();
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
    };
    int s = 0, sb = 0, rt = 0;
    // a finished row tile is stored ahead of the next step's requests: its stores are older than them for the wait
    auto next = [&]() {
        ++s;
        if (++sb == nb) {
            sb = 0;
            store_row_tile(rt++);
        }
    };
    while (s + 2 < n_steps) {
        step(s, sb, std::true_type{}, std::true_type{});
        next();
    }
    if (s + 1 < n_steps) {
        step(s, sb, std::true_type{}, std::false_type{});
        next();
    }
    step(s, sb, std::false_type{}, std::false_type{});
    next();
}

template <bool SWIGLU>
__global__ __launch_bounds__(kThreads, 2) void moe_stream_kernel(const MoeStreamArgs g) {
    extern __shared__ __align__(16) uint8_t smem[];
    // consecutive workgroups go round the 8 XCDs: all workgroups of a tile on one of them, so its activation rows come
    // into one L2
    const int x = (int)blockIdx.x & 7, k = (int)blockIdx.x >> 3, slot = k / g.wgs_per_tile * 8 + x, part = k % g.wgs_per_tile;
    const int4 tile = g.tiles[min(slot, g.list_capacity - 1)];   // (asked for together with the length of the list)
    if (slot >= *g.n_tiles) return;
    if (tile.z > 32) moe_stream_tile<SWIGLU, 2>(g, smem, tile, part);
    else moe_stream_tile<SWIGLU, 1>(g, smem, tile, part);
}

template <bool SWIGLU>
hipError_t launch(const MoeStreamArgs &g, unsigned wgs, hipStream_t s) {
    const int lds = moe_stream_lds(g.nb);
    static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&moe_stream_kernel<SWIGLU>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, moe_stream_lds(kMoeStreamMaxSb));
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL(moe_stream_kernel<SWIGLU>, dim3(wgs), dim3(kThreads), lds, s, g);
    return hipGetLastError();
}

}  // namespace

static_assert(moe_stream_lds(kMoeStreamMaxSb) <= 160 * 1024, "one workgroup's LDS");
static_assert(workgroups_per_cu(kMoeStreamMaxSb - 1) == 2, "two workgroups a compute unit up to 7936 weights a row");

bool moe_stream_fits(int type, int64_t K, int64_t N) {
    return type == kTypeQ4_K && K % 256 == 0 && K / 256 <= kMoeStreamMaxSb && N >= 1;
}

// t[0] (and t[1] = up when `swiglu`): Q4_K expert stacks; a.qs, a.d and a.hsum: the activation rows; args.active: the tile
// list of launch_moe_group with tile_rows = kMoeTileRows
hipError_t launch_moe_stream(const GemvArgs &args, int64_t n_pairs, bool swiglu, hipStream_t s) {
    const WeightView &w = args.t[0].w;
    if (!moe_stream_fits(w.type, w.K, w.N) || (swiglu && (args.t[1].w.type != w.type || args.t[1].w.K != w.K || args.t[1].w.N != w.N)) ||
        n_pairs < 1 || n_pairs > 0x7fffffff)
        return hipErrorInvalidValue;
    MoeStreamArgs g{};
    g.w0 = w.q4k;
    g.w1 = swiglu ? args.t[1].w.q4k : nullptr;
    g.y = args.t[0].y;
    g.qs = args.a.qs;
    g.d = args.a.d;
    g.hsum = args.a.hsum;
    g.order = args.order;
    const int64_t cap = moe_list_capacity(w.E, n_pairs, kMoeTileRows);
    g.tiles = reinterpret_cast<const int4 *>(args.active + active_slots_offset(cap));
    g.n_tiles = args.active + cap;
    g.list_capacity = (int)cap;
    g.N = w.N;
    g.nb = (int)(w.K / 256);
    g.x_div = args.x_div;
    const int64_t rows = kWaves * (swiglu ? 16 : 32), row_tiles = (w.N + rows - 1) / rows;
    // Row tiles a workgroup walks.  What a compute unit has to do, in steps of K: the workgroups it gets x their steps, and
    // about five more for every two workgroups (the start of a pipeline: list, pairs, rows, one trip to HBM after the
    // other), three where there is but one workgroup a compute unit to hide its waits, half as much again where its tiles are
    // full and it waits for arithmetic (8 experts of 4096 x 2048, 500 tokens: walking 3, 209 workgroups, 200 us, walking 1 147).  us a call, gate + up walking
    // 1 / 2 / 3 / 4 / 6 tiles: 128 experts of 2048 x 768, 64 tokens 92.4 / 96.7 / 89.7 / 99.3 / 95.7 (1536, 768, 512, 384, 256
    // workgroups); 32 experts of 4096 x 1536, 40 tokens 99 / 109 / 94 / 106 / 134; 2048 tokens over the 128 experts
    // 361 / 365 / 366 / 367 / 407.
    const int64_t busy = std::min<int64_t>(w.E, n_pairs);
    const int64_t expected = std::max<int64_t>(busy, busy / 2 + n_pairs / kMoeTileRows);   // tiles: the last one of an expert half full
    const int64_t cus = cu_count(), resident = workgroups_per_cu(g.nb);
    int64_t walk = 1, best = INT64_MAX;
    for (int64_t c = 1; c <= std::min<int64_t>(row_tiles, 64); ++c) {
        const int64_t per_cu = (expected * ((row_tiles + c - 1) / c) + cus - 1) / cus;
        const int64_t cost = per_cu * c * g.nb + 5 * ((per_cu + resident - 1) / resident) + (std::min(per_cu, resident) > 1 ? 0 : n_pairs > 16 * w.E ? c * g.nb / 2 : 3);
        if (cost < best) {
            best = cost;
            walk = c;
        }
    }
    walk = std::min<int64_t>(row_tiles, tuning_int(swiglu ? "QPROJ_MOE_STREAM_WALK" : "QPROJ_MOE_STREAM_WALK_DOWN", (int)walk));
    g.row_tiles = (int)walk;
    g.wgs_per_tile = (int)((row_tiles + walk - 1) / walk);
    const int64_t wgs = (cap + 7) / 8 * 8 * g.wgs_per_tile;
    if (wgs >= 0x7fffffff) return hipErrorInvalidValue;
    if (dry_run()) {
        plan_note("moe_stream_kernel<Q4_K%s>: tiles of up to %d pairs of an expert, %lld workgroups, %d a tile, %d row tiles of %lld each, %lld a compute unit", swiglu ? ", gate + up + swiglu" : "",
                  kMoeTileRows, (long long)wgs, g.wgs_per_tile, g.row_tiles, (long long)rows, (long long)resident);
        return hipSuccess;
    }
    if (!g.hsum || !args.order || !args.active) return hipErrorInvalidValue;
    return swiglu ? launch<true>(g, (unsigned)wgs, s) : launch<false>(g, (unsigned)wgs, s);
}

}  // namespace qproj
