// Q8_0 weights x ggml Q8_0 activation blocks on the int8 matrix cores in tiles of 96 or 64 tokens x 128 weight rows or 32
// tokens x 64: the batches that the 128 x 128 tiles of gemm_per32_kernel would fill with padding to a quarter and more, and matrices too small
// to fill the chip with those.
//
// Both operands change scale every 32 weights, so an int32 sum is valid for ONE matrix instruction and is folded into the
// fp32 sums right away: a float from the integer, the product of the two fp16 scales (exact), one fma.  Bound of the 96-token
// tiles: that vector work.  48 vector instructions a product, 53 with everything else; 3072 -> 2 x 8192 at 187 tokens keep the vector
// pipe busy 82 % of the launch, 8192 -> 3072 62 % (the matrix pipe 12 and 9).  The tiles of 32 tokens have 62 a product and wait as
// well, for the step's strip, its barrier and activations that are one step ahead only: 55 % busy for q/k/v of 3072 at 187 tokens,
// 37 % for o, a wave waiting for 36 % of its cycles.  So
//   - the weights are the rows of the matrix instruction, the tokens its columns: the scale of a token is one register a
//     token column, and the sixteen scales a lane needs of its weight rows are read once for all columns of the wave;
//   - a wave owns 32 weight rows of the tile and all of its tokens: its weights pass through a wave-private LDS strip straight
//     from global memory, two steps of 128 ahead (one: q/k/v of 3072 at 187 tokens, weights from HBM, 24.0 -> 29.5 us), and only the
//     activations are shared, one step ahead, one barrier a step;
//   - the requests to global memory go out one a product: in one go at the top of a step they hold up all waves of the workgroup
//     (3072 -> 2 x 8192 at 187 tokens 41.5 -> 37.6 us);
//   - the addend of the matrix instruction is the bits of 1.5 * 2^23, so its sums are floats already and a
//     subtraction (exact) takes the place of the conversion;
//   - K goes in two parts over the waves of a workgroup (KW = 2) while there is at most a workgroup a compute unit, the parts
//     meeting in LDS, and in stretches over workgroups (partial tiles, an adding pass) where the tiles leave units idle.
#include <algorithm>
#include <type_traits>

#include "gemm_convert.h"
#include "gemm_tiles.h"
#include "lds_direct.h"
#include "qproj_device.h"
#include "qproj_internal.h"

namespace qproj {

namespace {

constexpr int BK = 128;                 // weights of a row a step
constexpr int kStripBytes = 32 * BK + 256;   // 32 rows of codes, then their four fp16 scales a row
constexpr int kStripLoads = 5;
constexpr float kMagic = 12582912.f;    // 1.5 * 2^23: one integer step is one step of the float

struct Q8Target {
    const int8_t *qs;
    const uint16_t *d;
    float *out;                         // the output, or [n_split][M][N] partial tiles
    int64_t N;
    int tiles_n, tiles_pad, n_split, first_wg, vec4;   // tiles_pad: workgroups of one stretch, a multiple of the 8 XCDs
};
struct Q8Args {
    int n;
    Q8Target t[kMaxTargets];
    const int8_t *aq;
    const float *ad;
    int64_t M;
    int K, tiles_m;
};

// LDS: activations [2][KW][32 * WT tokens][128] (16-byte segments XOR-swizzled by the token), their scales
// [2][KW][tokens, 64 at a time][4], strips [2][wave], the scales of a step [wave][4][32] as floats
template <int WT, int KW, int RG>
struct Q8Lds {
    static constexpr int NW = RG * KW, kAct = WT * 4096, kDx = (WT + 1) / 2 * 1024;
    static constexpr int kOffDx = 2 * KW * kAct, kOffStrip = kOffDx + 2 * KW * kDx, kOffWs = kOffStrip + 2 * NW * kStripBytes,
                         kTotal = kOffWs + NW * 512;
    static_assert(kTotal <= 160 * 1024 / (KW == 1 || (WT == 1 && NW == 4) ? 2 : 1), "eight waves a compute unit");
    static_assert(KW == 1 || (WT + 1) / 2 * NW * 4096 <= kOffWs, "the K parts meet in the same LDS at the end");
};

// WT columns of 32 tokens, KW K parts, RG row groups of 32 weight rows.  TWO_LEVEL: shorter chains of sums.  The tiles of 32
// tokens take K whole, in chains of K / 64 blocks, where the 128-token tiles cut it in up to eight stretches: the sums of two steps
// are added up by themselves first, and their error is no larger.  The 96-token tiles set theirs aside in LDS halfway (a second set
// of 48 registers made the compiler pass its products through accumulator registers: 8 % slower).
template <int WT, int KW, int RG, bool TWO_LEVEL>
__global__ __launch_bounds__(64 * RG * KW, 2) void gemm_per32_kernel_q8_0(const Q8Args g) {
    using L = Q8Lds<WT, KW, RG>;
    constexpr int NW = L::NW, TM = 32 * WT;
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, lh = lane >> 5, rg = wave % RG, kp = wave / RG;

    Q8Target t = g.t[0];
#pragma unroll
    for (int i = 1; i < kMaxTargets; ++i)
        if (i < g.n && (int)blockIdx.x >= g.t[i].first_wg) t = g.t[i];
    const int local = (int)blockIdx.x - t.first_wg, split = local / t.tiles_pad, pid = local - split * t.tiles_pad;
    if (pid >= t.tiles_n * g.tiles_m) return;   // padding: the whole workgroup leaves
    int tile_n, tile_m;
    tile_of_workgroup(t.tiles_n, g.tiles_m, pid, tile_n, tile_m);
    const int64_t N = t.N, M = g.M, n0 = (int64_t)tile_n * (32 * RG) + rg * 32, m0 = (int64_t)tile_m * TM;
    const int K = g.K, nb = K / 32;
    // this workgroup's stretch, in units of 256; the two K parts take the steps of 128 in turn
    const int units = (K + 255) / 256, per = (units + t.n_split - 1) / t.n_split;
    const int ks_begin = min(split * per, units) * 2, ks_end = min(min((split + 1) * per, units) * 2, K / BK);
    const int n_steps = (ks_end - ks_begin + KW - 1) / KW;
    auto my_ks = [&](int s) { return min(ks_begin + s * KW + kp, ks_end - 1); };   // (past the end: any step, not added)

    // ---- weights: chunk c of a strip is its rows 8 c .. 8 c + 7; rows past the edge repeat the last one (never stored)
    const int64_t row0 = min(n0, N - 1);
    const int cap = (int)min(N - 1 - row0, (int64_t)31);
    const int8_t *const wbase = scalar_pointer(t.qs + row0 * K);
    const uint16_t *const dbase = scalar_pointer(t.d + row0 * nb);
    // slot lane % 8 of row r holds segment slot ^ (r / 2) % 8: 16 rows reading the same segment hit 16 different quadwords
    uint32_t woff[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int r = 8 * c + (lane >> 3);
        woff[c] = (uint32_t)min(r, cap) * (uint32_t)K + 16u * ((lane & 7) ^ ((r >> 1) & 7));
    }
    const uint32_t doff = (uint32_t)min(lane >> 1, cap) * (uint32_t)nb + 2u * (lane & 1);
    uint8_t *const strip = smem + L::kOffStrip + wave * kStripBytes;   // second buffer NW * kStripBytes further on
    auto request_strip = [&](int s, uint8_t *dst) {
        const uint32_t ks = (uint32_t)my_ks(s);
#pragma unroll
        for (int c = 0; c < 4; ++c) global_to_lds16(wbase + (woff[c] + ks * BK), dst + 1024 * c);
        global_to_lds4(dbase + (doff + ks * 4u), dst + 4096);
    };

    // ---- activations of a K part: request j of a wave = tokens 8 (rg + RG j) .. +7; scales: 64 tokens a request
    const int mcap = (int)min(M - 1 - m0, (int64_t)TM - 1);
    const int8_t *const abase = scalar_pointer(g.aq + m0 * K);
    const float *const xbase = scalar_pointer(g.ad + m0 * nb);
    constexpr int AR = 4 * WT / RG;
    uint32_t aoff[AR];
#pragma unroll
    for (int j = 0; j < AR; ++j) {
        const int r = 8 * (rg + RG * j) + (lane >> 3);
        aoff[j] = (uint32_t)min(r, mcap) * (uint32_t)K + 16u * ((lane & 7) ^ ((r >> 1) & 7));
    }
    const int xg = rg % ((WT + 1) / 2);   // (the other waves ask for the same once more: no branch in the step)
    const uint32_t xoff = (uint32_t)min(xg * 64 + lane, mcap) * (uint32_t)nb;
    auto request_acts = [&](int s) {
        const uint32_t ks = (uint32_t)my_ks(s);
        const int buf = (s & 1) * KW + kp;
#pragma unroll
        for (int j = 0; j < AR; ++j) global_to_lds16(abase + (aoff[j] + ks * BK), smem + buf * L::kAct + (rg + RG * j) * 1024);
        global_to_lds16(xbase + (xoff + ks * 4u), smem + L::kOffDx + buf * L::kDx + xg * 1024);
    };

    float sum[WT][16], total[WT == 1 ? 16 : 1];
#pragma unroll
    for (int j = 0; j < WT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) sum[j][v] = 0.f;
    if constexpr (WT == 1) {
#pragma unroll
        for (int v = 0; v < 16; ++v) total[v] = 0.f;
    }
    v4i *const aside = reinterpret_cast<v4i *>(smem + L::kTotal + wave * (WT * 4096)) + lane;
    auto fold_sums = [&]() {
        if constexpr (TWO_LEVEL) {
#pragma unroll
            for (int j = 0; j < WT; ++j) {
                if constexpr (WT > 1) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        aside[(4 * j + i) * 64] = v4i{__float_as_int(sum[j][4 * i]), __float_as_int(sum[j][4 * i + 1]), __float_as_int(sum[j][4 * i + 2]),
                                                      __float_as_int(sum[j][4 * i + 3])};
                }
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    if constexpr (WT == 1) total[v] += sum[0][v];
                    sum[j][v] = 0.f;
                }
            }
        }
    };
    auto add_folded = [&](int n_steps) {
        if constexpr (TWO_LEVEL && WT == 1) {
#pragma unroll
            for (int v = 0; v < 16; ++v) sum[0][v] += total[v];
        } else if constexpr (TWO_LEVEL) {
            if (n_steps >= 3) {
#pragma unroll
                for (int j = 0; j < WT; ++j)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const v4i o = aside[(4 * j + i) * 64];
#pragma unroll
                        for (int r = 0; r < 4; ++r) sum[j][4 * i + r] += __int_as_float(o[r]);
                    }
            }
        }
    };
    v16i addend;
#pragma unroll
    for (int v = 0; v < 16; ++v) addend[v] = __float_as_int(kMagic);
    asm volatile("" : "+v"(addend));   // in registers: rebuilt for every product it costs eight moves
    float *const ws_tab = reinterpret_cast<float *>(smem + L::kOffWs + wave * 512);
    // segment 2 * kb + lh of row l32 (of the strip, of a token tile): offset ^ 32 * kb
    const int foff = l32 * BK + 16 * (lh ^ ((l32 >> 1) & 7));

    auto step = [&](int s, auto more1, auto more2) {
        constexpr bool MORE1 = decltype(more1)::value, MORE2 = decltype(more2)::value;
        uint8_t *const sbuf = strip + (s & 1) * NW * kStripBytes;
        v4i wf[4];
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) wf[kb] = *reinterpret_cast<const v4i *>(sbuf + (foff ^ (32 * kb)));
        const uint32_t d2 = *reinterpret_cast<const uint32_t *>(sbuf + 4096 + l32 * 8 + 4 * lh);   // blocks 2 lh, 2 lh + 1 of row l32
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the strip has been read: it may be overwritten
        // The requests go out one a product, the activations first: sent in one go at the top of a step they stall each
        // other (a compute unit takes 64 bytes of them a cycle) and leave the SIMDs to one wave.
        auto request = [&](int i) {
            if (MORE1 && i <= AR) {
                const uint32_t ks = (uint32_t)my_ks(s + 1);
                const int buf = ((s + 1) & 1) * KW + kp;
                if (i < AR) global_to_lds16(abase + (aoff[i < AR ? i : 0] + ks * BK), smem + buf * L::kAct + (rg + RG * i) * 1024);
                else global_to_lds16(xbase + (xoff + ks * 4u), smem + L::kOffDx + buf * L::kDx + xg * 1024);
            } else if (MORE2 && i > AR && i <= AR + kStripLoads) {
                const uint32_t ks = (uint32_t)my_ks(s + 2);
                const int c = i - AR - 1;
                if (c < 4) global_to_lds16(wbase + (woff[c < 4 ? c : 0] + ks * BK), sbuf + 1024 * c);
                else global_to_lds4(dbase + (doff + ks * 4u), sbuf + 4096);
            }
        };
        __builtin_amdgcn_sched_barrier(0);
        constexpr int kRequests = AR + 1 + kStripLoads, kProducts = 4 * WT;
        auto requests_of = [&](int q) {   // those that go with product q
#pragma unroll
            for (int i = q * kRequests / kProducts; i < (q + 1) * kRequests / kProducts; ++i) request(i);
        };
        const bool live = KW == 1 || ks_begin + s * KW + kp < ks_end;
        if (live) {
            ws_tab[(2 * lh) * 32 + l32] = h2f(d2);
            ws_tab[(2 * lh + 1) * 32 + l32] = h2f(d2 >> 16);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            const int buf = (s & 1) * KW + kp;
            const uint8_t *const ab = smem + buf * L::kAct, *const xb = smem + L::kOffDx + buf * L::kDx;
            v4i dx[WT];   // the token's four scales
#pragma unroll
            for (int j = 0; j < WT; ++j) dx[j] = *reinterpret_cast<const v4i *>(xb + (j * 32 + l32) * 16);
            // Pinned product by product: the next one's matrix instruction goes out ahead of this one's fold, the operands of
            // the next 32 weights are read during the fold of this block's first.
            v4i ws[2][4], af[2][WT];
            v16i I[2];
            auto load = [&](int kb) {
#pragma unroll
                for (int j = 0; j < WT; ++j) af[kb & 1][j] = *reinterpret_cast<const v4i *>(ab + j * 4096 + (foff ^ (32 * kb)));
#pragma unroll
                for (int i = 0; i < 4; ++i) ws[kb & 1][i] = *reinterpret_cast<const v4i *>(ws_tab + kb * 32 + 8 * i + 4 * lh);
            };
            auto multiply = [&](int q) {
                I[q & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[q / WT], af[(q / WT) & 1][q % WT], addend, 0, 0, 0);
            };
            load(0);
            multiply(0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < 4 * WT; ++q) {
                const int kb = q / WT, j = q % WT;
                if (j == 0 && kb < 3) load(kb + 1);
                if (WT == 1) __builtin_amdgcn_sched_barrier(0);
                if (q + 1 < 4 * WT) multiply(q + 1);
                requests_of(q);
                __builtin_amdgcn_sched_barrier(0);
                const float da = __int_as_float(dx[j][kb]);
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    sum[j][v] = fmaf(__int_as_float(I[q & 1][v]) - kMagic, __int_as_float(ws[kb & 1][v >> 2][v & 3]) * da, sum[j][v]);
                // (left alone the compiler postpones the last fma of every output and spills)
#pragma unroll
                for (int v = 0; v < 16; ++v) asm volatile("" : "+v"(sum[j][v]));
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        } else {
#pragma unroll
            for (int q = 0; q < kProducts; ++q) requests_of(q);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (MORE1) {
            if constexpr (MORE2) wait_vmcnt<kStripLoads>();   // all but the strip just asked for
            else wait_vmcnt<0>();
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
    };
    if (n_steps > 0) {
        request_strip(0, strip);
        request_acts(0);
        request_strip(1, strip + NW * kStripBytes);   // (of a single step: once more)
        wait_vmcnt<kStripLoads>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        int s = 0;
        for (; s + 2 < n_steps; ++s) {
            step(s, std::true_type{}, std::true_type{});
            if (WT == 1 ? (s & 1) != 0 : s + 1 == n_steps / 2) fold_sums();   // (of three steps and more)
        }
        if (s + 1 < n_steps) step(s++, std::true_type{}, std::false_type{});
        step(s, std::false_type{}, std::false_type{});
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (a single step leaves its second strip request behind)
    add_folded(n_steps);

    // ---- the K parts meet in LDS: part q keeps token tiles j % 2 == q, the other hands its sums over
    if constexpr (KW == 2) {
        __syncthreads();
        v4i *const meet = reinterpret_cast<v4i *>(smem);
#pragma unroll
        for (int j = 0; j < WT; ++j)
            if (j % 2 != kp) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    meet[((wave * ((WT + 1) / 2) + j / 2) * 4 + i) * 64 + lane] = v4i{__float_as_int(sum[j][4 * i]), __float_as_int(sum[j][4 * i + 1]),
                                                                                    __float_as_int(sum[j][4 * i + 2]), __float_as_int(sum[j][4 * i + 3])};
            }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < WT; ++j)
            if (j % 2 == kp) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const v4i o = meet[((((kp ^ 1) * RG + rg) * ((WT + 1) / 2) + j / 2) * 4 + i) * 64 + lane];
#pragma unroll
                    for (int r = 0; r < 4; ++r) sum[j][4 * i + r] += __int_as_float(o[r]);   // two addends: either order
                }
            }
    }
    // ---- store: register v of lane l is weight row 8 (v / 4) + 4 (l / 32) + v % 4, token l % 32
    float *const out = t.out + (size_t)split * M * N;
#pragma unroll
    for (int j = 0; j < WT; ++j) {
        if (KW == 2 && j % 2 != kp) continue;
        const int64_t m = m0 + j * 32 + l32;
        if (m >= M) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t n = n0 + 8 * i + 4 * lh;
            float *const o = out + m * N + n;
            if (t.vec4) {   // rows of whole, aligned float4s
                if (n < N) *reinterpret_cast<float4 *>(o) = make_float4(sum[j][4 * i], sum[j][4 * i + 1], sum[j][4 * i + 2], sum[j][4 * i + 3]);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n + r < N) o[r] = sum[j][4 * i + r];
            }
        }
    }
}

struct Q8Plan {
    int wt, kw, n_split;
    bool one_round;   // of workgroups, one a compute unit (two K parts)
    bool two_level;   // in workgroups of 64 rows, the sums added up in two levels
};

// q, k, v and o: square matrices and small ones, whose launch holds a matrix and a half of K rows as a rule
bool rider(int64_t K, int64_t N) { return K == N || N <= 1024; }
int64_t rider_tiles(int64_t K, int64_t M) { return (M + 31) / 32 * ((K + K / 2 + 127) / 128); }

// Tile and cut of a matrix this kernel takes, by the matrix and the row count alone (the bits of its results do not depend on
// what rides along).
Q8Plan q8_plan(int64_t K, int64_t M, int64_t N) {
    const int64_t cus = cu_count(), units = (K + 255) / 256;
    Q8Plan p{};
    p.wt = tuning_int("QPROJ_Q8_WT", rider(K, N) ? 1 : M <= 64 ? 2 : 3);
    const int64_t tiles_m = (M + 32 * p.wt - 1) / (32 * p.wt);
    // workgroups of a stretch, the same number on each of the 8 XCDs: 8192 -> 2304 at 160 tokens is 36 tiles, five on four of
    // the XCDs; seven stretches of them are 252 workgroups, but 35 for the 32 units of those (32.8 us in 128-token tiles, 39.5 in
    // seven stretches, 30.5 in six)
    const int64_t stretch = (tiles_m * ((N + 127) / 128) + 7) / 8 * 8;
    // (a matrix taller than its rows are long has a sibling in the launch as a rule: up beside gate)
    const int64_t tiles = rider(K, N) ? rider_tiles(K, M) : N > K ? 2 * stretch : stretch;
    // Up to a workgroup a compute unit K goes in two parts inside the workgroup, and in stretches that fill the chip once; beyond
    // that workgroups of four waves share a compute unit out of step (3072 -> 2 x 8192 at 187 tokens 37.6 against 44.9 us, 4096 ->
    // 2 x 14336 122 either way).  The tiles of 32 and 64 tokens are built with two parts only:
    // q8_0_tokens_takes leaves their larger grids to the 128-token tiles.
    p.kw = tuning_int("QPROJ_Q8_KW", p.wt >= 3 && tiles > cus ? 1 : 2);
    int64_t n = std::max<int64_t>(1, std::min<int64_t>(8, cus / tiles));
    // never longer sums than the 128 x 128 tiles have (their error against 64 bits grows with the length; two levels of them instead
    // in the tiles of 32 tokens)
    const int64_t least = p.wt > 1 ? (per32_splits(kTypeQ8_0, K, M, N) + p.kw - 1) / p.kw : 1;
    p.two_level = p.wt == 1;
    const auto tidy = [&](int64_t parts) {
        parts = std::max<int64_t>(1, std::min<int64_t>(parts, units / 2));   // two times 256 weights a stretch at least
        if ((M * N) % 4 != 0) parts = 1;
        while (parts > 1 && (units + parts - 2) / (parts - 1) == (units + parts - 1) / parts) --parts;   // no stretch without work
        return parts;
    };
    n = tidy(tuning_int("QPROJ_Q8_SPLIT", (int)std::max<int64_t>(n, least)));
    // Where that leaves a workgroup two to four steps, most of it the start of a pipeline, about half as many stretches in workgroups
    // of half the rows, still one round, walk twice as far, their sums in two levels (error against 64 bits 0.68 to 0.94 of the
    // 128-token tiles'; up to 1.02 of the short stretches').  us a call, 128-token tiles / eight waves, short stretches / four waves:
    // 3072 -> 1536 at 160 tokens 19.2 / 21.1 / 17.5, 4096 -> 1280 20.6 / 21.7 / 18.9, 3584 -> 2304 26.9 / 32.3 / 23.7, 5120 -> 1280 23.6 /
    // 23.5 / 20.2; 4096 -> 3072 at 80 21.4 / 21.8 / 19.1, 8192 -> 4096 28.1 / 27.4 / 26.6.  (Stretches that are one round in such workgroups
    // as they are get them from the launcher and stay as they are: two levels would cost 4 % there.)
    if (p.wt == 3 && p.kw == 2 && K > N && !rider(K, N) && (units + n - 1) / n <= 4) {
        const int64_t half_stretch = (tiles_m * ((N + 63) / 64) + 7) / 8 * 8, halves = cus / half_stretch;
        if (n * half_stretch > cus && halves >= least) {
            n = tidy(std::min<int64_t>(8, halves));
            p.two_level = true;
        }
    }
    p.n_split = (int)n;
    p.one_round = tiles * n <= cus;
    return p;
}

size_t partial_bytes(const Q8Plan &p, int64_t M, int64_t N) { return p.n_split > 1 ? (size_t)p.n_split * M * N * 4 : 0; }

template <int WT, int KW, int RG, bool TWO_LEVEL>
hipError_t launch(const Q8Args &g, int wgs, hipStream_t s) {
    constexpr int lds = Q8Lds<WT, KW, RG>::kTotal + (TWO_LEVEL && WT > 1 ? RG * KW * WT * 4096 : 0);
    static_assert(lds <= 160 * 1024, "one workgroup's LDS");
    const auto kern = &gemm_per32_kernel_q8_0<WT, KW, RG, TWO_LEVEL>;
    static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(64 * RG * KW), lds, s, g);
    return hipGetLastError();
}

using LaunchFn = hipError_t (*)(const Q8Args &, int, hipStream_t);
LaunchFn instance(int wt, int kw, int rg, bool two_level) {   // null: not built
#define QP_Q8(WT, KW, RG, TWO_LEVEL) \
    if (wt == WT && kw == KW && rg == RG && two_level == TWO_LEVEL) return &launch<WT, KW, RG, TWO_LEVEL>
    QP_Q8(1, 2, 2, true);
    QP_Q8(2, 2, 4, false);
    QP_Q8(3, 1, 4, false);
    QP_Q8(3, 2, 4, false);
    QP_Q8(3, 2, 2, false);
    QP_Q8(3, 2, 2, true);
#ifdef QPROJ_TUNING
    QP_Q8(1, 2, 4, true);
    QP_Q8(1, 1, 4, true);
    QP_Q8(2, 1, 4, false);
    QP_Q8(4, 1, 4, false);
    QP_Q8(4, 2, 4, false);
#endif
#undef QP_Q8
    return nullptr;
}

}  // namespace

// Which products this kernel takes from the 128 x 128 tiles: of those where a 128-token tile is padding for a quarter and more
// and the tiles of 96 or 64 tokens are not, 129 .. 192 tokens, and rows longer than the matrix is tall up to 96 tokens.
// us a call at 160 tokens, 128-token tiles / here: 3072 -> 2 x 8192 50.3 / 39.2, 4096 -> 2 x 14336 96 / 80, 4096 -> 32000 100 / 84,
// 8192 -> 3072 38.0 / 33.4, 14336 -> 4096 66.2 / 52.3, 28672 -> 8192 210 / 143; at 64 tokens 8192 -> 3072 26.4 / 23.8, 28672 -> 8192
// 114 / 86.  Not 1024 -> 2 x 2816 (19.1 / 19.9).
// Square and small matrices take tiles of 32 tokens while they are one round of workgroups: the grid is filled with few
// stretches of K or none, so the partial tiles and their adding pass go.  q/k/v with 512 (2048) and 1024 rows for k and v: of 2048 at
// 33 / 128 / 250 tokens 16.6 / 13.2, 19.6 / 16.0, 23.6 / 17.8, of 3072 at 64 / 187 21.7 / 17.6, 30.7 / 24.3, of 4096 at 64 27.0 / 22.1.  Left slower, by up to 9 %: launches a little beyond a round,
// q/k/v of 3072 with 1024 for k and v at 193 .. 224 tokens (30.9 / 33.6), of 2560 at 97 .. 128 (21.8 / 23.5), three of 3072 at 80.
// Gate and up whose sums have to be cut to be as short as those of the 128-token tiles, so that they are two rounds of workgroups,
// stay there: 2048 -> 2 x 5120 at 160 tokens 33.4 / 41.9, 1536 -> 2 x 4608 at 192 29.6 / 39.5.
// Not taken, though measured faster here: gate and up at 33 .. 96 tokens (3072 -> 2 x 8192 at 33 / 64 / 96 32.2 / 25.3, 34.6 / 28.2, 36.6 /
// 33.6, 4096 -> 2 x 14336 at 48 60.8 / 42.3), 257 .. 288 tokens (4096 -> 2 x 14336 147 / 129, 14336 -> 4096 101 / 74), squares beyond 64
// tokens: 3072 at 128 21.5 / 18.0, 3584 at 97 / 160 22.1 / 19.6, 27.3 / 22.1, 4096 at 128 / 160 24.1 / 22.2, 29.0 / 25.1 (as q/k/v at
// 192, beyond a round, 36.8 / 43.6).
bool q8_0_tokens_takes(int64_t K, int64_t M, int64_t N) {
    if (K % BK != 0 || K > (1 << 24)) return false;   // 32-bit lane offsets: 128 rows of K bytes
    if (tuning_int("QPROJ_Q8_TAKE", 0)) return true;
    if (K <= 1024) return false;
    const int64_t cus = cu_count();
    if (rider(K, N)) return (K <= 3072 && rider_tiles(K, M) * (M > 128 ? 1 : 2) <= cus) || (K <= 4096 && M <= 64 && rider_tiles(K, M) <= cus);
    if (M > 128 && M <= 192) {
        const Q8Plan p = q8_plan(K, M, N);
        return p.kw == 1 || p.one_round;
    }
    return M > 32 && M <= 96 && K > N && N <= 128 * cus;
}

size_t q8_0_tokens_scratch_bytes(int64_t K, int64_t M, int64_t N) { return partial_bytes(q8_plan(K, M, N), M, N); }

// Q8_0 weights x ggml Q8_0 activation blocks (planes in `a`).  A launch takes as many of the matrices as have room for their
// partial tiles in the scratch and share the shape of the workgroups; the next launch uses the same bytes again, behind the
// adding pass.
hipError_t launch_gemm_q8_0_tokens(int n, const WeightView *w, const ActView &a, int64_t M, float *const *y, const Scratch &sc, hipStream_t s) {
    if (n < 1 || n > kMaxTargets || a.kind != kActKindQ8_0 || M <= 0) return hipErrorInvalidValue;
    Q8Plan plans[kMaxTargets];
    for (int i = 0; i < n; ++i) {
        if (w[i].type != kTypeQ8_0 || w[i].K != w[0].K || !q8_0_tokens_takes(w[i].K, M, w[i].N)) return hipErrorInvalidValue;
        plans[i] = q8_plan(w[i].K, M, w[i].N);
        if (!sc.p) plans[i].n_split = 1;
    }
    for (int first = 0; first < n;) {
        Q8Args g{};
        g.aq = a.qs;
        g.ad = a.d;
        g.M = M;
        g.K = (int)w[0].K;
        const Q8Plan &p0 = plans[first];
        const int64_t tiles_m = (M + 32 * p0.wt - 1) / (32 * p0.wt);
        const auto shares = [&](int i) { return plans[i].kw == p0.kw && plans[i].wt == p0.wt && plans[i].two_level == p0.two_level; };
        const auto tiles_pad = [&](int i, int rows) { return ((w[i].N + rows - 1) / rows * tiles_m + 7) / 8 * 8; };
        // Half the weight rows a workgroup where that many workgroups are still one a compute unit: the same sums on twice the
        // compute units (a matrix is cut as if its sibling rode along; 3072 -> 8192 alone at 187 tokens 35.0 -> 27.8 us).
        int64_t halves = 0;
        for (int i = first; i < n && shares(i); ++i) halves += tiles_pad(i, 64) * plans[i].n_split;
        // Tiles of 32 tokens always: two workgroups of four waves share a compute unit (56 KB of LDS each) and hide each other's
        // barriers, and q/k/v a little beyond a round of eight-wave workgroups do not take two.  us a call, tiles of 128 tokens / 128
        // rows a workgroup / 64: q/k/v of 2560 with 1024 for k and v at 97 tokens 21.8 / 28.0 / 23.5, of 3072 at 187 30.7 / 25.1 / 24.3
        // and at 193 30.9 / 38.6 / 33.6, three of 2048 at 80 21.0 / 24.5 / 21.9; 3072 -> 1024 alone at 187 18.8 / 22.4 / 17.8.
        const int rg = tuning_int("QPROJ_Q8_RG", p0.two_level || (p0.wt == 3 && p0.kw == 2 && halves <= cu_count()) ? 2 : 4);
        const LaunchFn run = instance(p0.wt, p0.kw, rg, p0.two_level);
        if (!run) return hipErrorInvalidValue;   // (in a dry run too)
        SumTargets sums{};
        size_t used = 0;
        int64_t wg = 0;
        int i = first;
        for (; i < n && shares(i); ++i) {
            const Q8Plan &p = plans[i];
            const size_t bytes = partial_bytes(p, M, w[i].N);
            const int64_t pad = tiles_pad(i, 32 * rg);
            if ((used + bytes > sc.bytes && bytes) || wg + pad * p.n_split >= 0x7fffffff) {
                if (i == first) return hipErrorInvalidValue;   // partial tiles would not fit
                break;
            }
            Q8Target &t = g.t[g.n++];
            t.qs = w[i].q8_qs;
            t.d = w[i].q8_d;
            t.out = y[i];
            t.N = w[i].N;
            if (bytes) {
                if (!dry_run()) t.out = sc.p + used / 4;
                add_sum(sums, t.out, y[i], p.n_split, M * w[i].N);
                used += bytes;
            }
            t.vec4 = w[i].N % 4 == 0 && (reinterpret_cast<uintptr_t>(t.out) & 15) == 0;
            t.tiles_n = (int)((w[i].N + 32 * rg - 1) / (32 * rg));
            t.tiles_pad = (int)pad;
            t.n_split = p.n_split;
            t.first_wg = (int)wg;
            wg += pad * p.n_split;
            if (dry_run())
                plan_note("gemm_per32_kernel_q8_0<%d token tiles, %d K parts>%s: tile %d tokens x %d rows, %lld tiles x %d K stretches%s%s", p.wt, p.kw,
                          g.n > 1 ? " (same launch)" : "", 32 * p.wt, 32 * rg, (long long)(t.tiles_n * tiles_m), p.n_split,
                          p.wt > 1 && p.two_level ? " of two levels of sums" : "", p.n_split > 1 ? " + sum_parts_kernel" : "");
        }
        first = i;
        g.tiles_m = (int)tiles_m;
        if (dry_run()) {
            if (sums.n) plan_note_cut();
            continue;
        }
        hipError_t e = run(g, (int)wg, s);
        if (e == hipSuccess && sums.n) e = launch_sum_parts(sums, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace qproj
