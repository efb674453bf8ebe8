// Batches between the small-batch kernel and the wide prefill tiles, and matrices too small for those: weights streamed
// from HBM once for up to 128 tokens, Q4_K / Q6_K weights x ggml Q8_K activations on the int8 matrix cores.
//
// Bound on paper: HBM (33 .. ~100 tokens).  Measured, no unit alone: gate + up of 14336 rows at 48 tokens move 68.3 MB (the
// weights once) in 28.4 us = 2.4 TB/s, the vector pipe busy a third and the matrix pipe a quarter of the cycles, a wave waiting
// for 39 % of its own.  What kept the 64-token tiles further below (49 us there) was latency, not arithmetic: one
// super-block of weights in flight a wave, a launch a matrix, too few workgroups.  So here
//   - raw weight blocks go from global memory straight into wave-private LDS strips, two super-blocks ahead of the
//     arithmetic (Q4_K; one ahead for the larger Q6_K strips): a wave reads its strip into registers at the top of a
//     step and asks for the block after next into the same strip, so 8 waves keep 2 x 37 KB a compute unit in flight;
//   - activations of a step (one super-block a K part) are double-buffered in LDS, shared by the row groups of the
//     workgroup, one barrier a step;
//   - a workgroup is 8 waves (4 where the launch leaves room for twice the workgroups) = RW row groups of 32 weight
//     rows x KW K parts (summed through LDS at the end), K is cut further over workgroups where the tiles would not
//     fill the chip, and all matrices of a call (q/k/v, gate/up) share the launch and the launch that adds the partial
//     tiles.
// The arithmetic is that of the tiled kernels: Q4_K scales in base 8 as two int8 operands, Q6_K products as high and
// low bytes, both chains inside the matrix cores for a whole super-block, one flush per 256 weights, the Q4_K min
// term on the fp16 cores from the plane the quantizer wrote.
#include <limits.h>
#include <stddef.h>
#include <stdlib.h>

#include <algorithm>

#include "gemm_convert.h"
#include "gemm_tiles.h"
#include "lds_direct.h"
#include "qproj_device.h"
#include "qproj_internal.h"

namespace qproj {

namespace {

struct StreamTarget {
    const uint8_t *p0, *p1, *p2, *p3;   // Q4_K: blocks; Q6_K: ql, qh, scales, d
    float *out;                         // [n_split][M][N] partial tiles, or the output itself when K is whole
    int N, tiles_n, tiles_pad, n_split; // tiles_pad: workgroups of one stretch of K (a multiple of 8)
};

// By field: arguments come a 64-byte line at a time, a trip to memory each, and Q4_K needs three of these lines; all of them are
// asked for at once.  us a call, quantizer included, on one card: 4096 x 4096 at 48 tokens 16.5 -> 16.0, 4096 -> 28672 29.6 -> 28.8, at
// 96 tokens 19.4 -> 18.9 and 45.7 -> 45.2; Q6_K level to 2 %.
struct StreamArgs {
    const int8_t *qs;                   // activations
    const float *d;
    const uint16_t *msum;
    const float *rs;
    int M, nb, tiles_m;
    int first_wg[kMaxTargets];          // of the launch's matrices; INT_MAX where there is none
    int N[kMaxTargets], tiles_n[kMaxTargets], tiles_pad[kMaxTargets], n_split[kMaxTargets];
    float *out[kMaxTargets];
    const uint8_t *p0[kMaxTargets];
    const uint8_t *p1[kMaxTargets], *p2[kMaxTargets], *p3[kMaxTargets];
};

template <int QT>
struct Strip;

// 32 rows x 144 bytes as they lie in memory (row stride 144 B: conflict-free 16-byte reads): 288 pieces, the last
// half-filled request repeats piece 287
template <>
struct Strip<kTypeQ4_K> {
    static constexpr int kBytes = 5 * 1024, kLoads = 5;
    struct Raw {
        v4i hdr, q[4];
    };
    const uint8_t *base;
    uint32_t off[5];
    __device__ __forceinline__ void init(const StreamTarget &t, int nb, int64_t row0, int cap, int lane) {
        base = scalar_pointer(t.p0 + row0 * nb * 144);
#pragma unroll
        for (int c = 0; c < 5; ++c) {
            const int p = min(lane + 64 * c, 287);
            off[c] = (uint32_t)(min(p / 9, cap) * nb * 144 + 16 * (p % 9));
        }
    }
    __device__ __forceinline__ void request(uint32_t sb, uint8_t *strip, int c) const { global_to_lds16(base + (off[c] + sb * 144u), strip + 1024 * c); }
    static __device__ __forceinline__ Raw read(const uint8_t *strip, int l32, int lh) {
        Raw r;
        r.hdr = *reinterpret_cast<const v4i *>(strip + l32 * 144);
#pragma unroll
        for (int i = 0; i < 4; ++i) r.q[i] = *reinterpret_cast<const v4i *>(strip + l32 * 144 + 16 + 64 * lh + 16 * i);
        return r;
    }
};

// ql [row][8 slots], qh [row][4 slots] and the 16 scales of a row: a load straight into LDS cannot pad rows, so the
// 16-byte pieces of a row are permuted by the row index (any 16 consecutive rows reading the same piece hit 16
// different slots)
template <>
struct Strip<kTypeQ6_K> {
    static constexpr int kBytes = 7 * 1024, kLoads = 7;
    struct Raw {
        v4i ql[4], qh[2];   // [2*gl + e], [e]
        v2i sc;
    };
    const uint8_t *bl, *bh, *bs;
    global_ptr<uint16_t> bd;
    uint32_t off_l[4], off_h[2], off_s, off_d;
    static __device__ __forceinline__ int xl(int r) { return ((r >> 1) & 3) | (((r ^ (r >> 3)) & 1) << 2); }
    static __device__ __forceinline__ int xh(int r) { return ((r >> 2) & 1) | ((((r >> 1) ^ (r >> 3)) & 1) << 1); }
    __device__ __forceinline__ void init(const StreamTarget &t, int nb, int64_t row0, int cap, int lane) {
        bl = scalar_pointer(t.p0 + row0 * nb * 128);
        bh = scalar_pointer(t.p1 + row0 * nb * 64);
        bs = scalar_pointer(t.p2 + row0 * nb * 16);
        bd = scalar_global(reinterpret_cast<const uint16_t *>(t.p3) + row0 * nb);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int p = lane + 64 * c, r = p >> 3;
            off_l[c] = (uint32_t)(min(r, cap) * nb * 128 + 16 * ((p & 7) ^ xl(r)));
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int p = lane + 64 * c, r = p >> 2;
            off_h[c] = (uint32_t)(min(r, cap) * nb * 64 + 16 * ((p & 3) ^ xh(r)));
        }
        off_s = (uint32_t)(min(lane & 31, cap) * nb * 16);
        off_d = (uint32_t)(min(lane & 31, cap) * nb);
    }
    __device__ __forceinline__ void request(uint32_t sb, uint8_t *strip, int c) const {
        if (c < 4) global_to_lds16(bl + (off_l[c & 3] + sb * 128u), strip + 1024 * c);
        else if (c < 6) global_to_lds16(bh + (off_h[c & 1] + sb * 64u), strip + 1024 * c);
        else global_to_lds16(bs + (off_s + sb * 16u), strip + 6144);   // the upper half lands behind: not read
    }
    __device__ __forceinline__ uint32_t scale(uint32_t sb) const { return load_global<uint16_t>(bd, 2u * (off_d + sb)); }
    static __device__ __forceinline__ Raw read(const uint8_t *strip, int l32, int lh) {
        Raw r;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
#pragma unroll
            for (int gl = 0; gl < 2; ++gl)
                r.ql[2 * gl + e] = *reinterpret_cast<const v4i *>(strip + l32 * 128 + 16 * ((4 * lh + 2 * gl + e) ^ xl(l32)));
            r.qh[e] = *reinterpret_cast<const v4i *>(strip + 4096 + l32 * 64 + 16 * ((2 * lh + e) ^ xh(l32)));
        }
        r.sc = *reinterpret_cast<const v2i *>(strip + 6144 + l32 * 16 + 8 * lh);
        return r;
    }
};

// LDS of a workgroup: [2][KW] activation tiles (32 * JT tokens x 256, 16-byte segments XOR-swizzled by the token),
// [2][KW] min-term tiles (Q4_K), the scales of kScaleSb super-blocks (activations [super-block][token]; Q6_K weights
// [wave][super-block][row]), then the strips
template <int QT, int JT, int KW, int SW, int NW>
struct StreamLds {
    static constexpr int kScaleSb = JT <= 2 ? 16 : 8;
    static constexpr int kAct = JT * 8192, kMs = QT == kTypeQ4_K ? JT * 1024 : 0, kDx = JT * 128;
    static constexpr int kDwWave = QT == kTypeQ6_K ? kScaleSb / KW * 64 : 0;
    static constexpr int kOffMs = 2 * KW * kAct, kOffDx = kOffMs + 2 * KW * kMs, kOffDw = kOffDx + kScaleSb * kDx,
                         kOffStrip = kOffDw + NW * kDwWave;
    static constexpr int kTotal = kOffStrip + NW * SW * Strip<QT>::kBytes;
    static_assert(kTotal <= 160 * 1024, "one workgroup's LDS");
    static_assert(NW * JT * 4096 <= kOffStrip || KW == 1, "the K parts meet in the same LDS at the end");
};

template <int QT, int JT, int KW, int SW, int NW>
__global__ __launch_bounds__(64 * NW, 1) void gemm_stream_kernel(const StreamArgs g) {
    using S = Strip<QT>;
    using L = StreamLds<QT, JT, KW, SW, NW>;
    constexpr bool kQ4 = QT == kTypeQ4_K;
    constexpr int RW = NW / KW, TM = 32 * JT, NT = 64 * NW;
    extern __shared__ __align__(16) uint8_t smem[];
    fetch_arguments<decltype(gemm_stream_kernel<QT, JT, KW, SW, NW>), kQ4 ? offsetof(StreamArgs, p1) : sizeof(StreamArgs)>();
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, lh = lane >> 5, rg = wave % RW, kp = wave / RW;

    int ti = 0;
#pragma unroll
    for (int i = 1; i < kMaxTargets; ++i)
        if ((int)blockIdx.x >= g.first_wg[i]) ti = i;
    const StreamTarget t = {g.p0[ti], kQ4 ? nullptr : g.p1[ti], kQ4 ? nullptr : g.p2[ti], kQ4 ? nullptr : g.p3[ti],
                            g.out[ti], g.N[ti], g.tiles_n[ti], g.tiles_pad[ti], g.n_split[ti]};
    const int local = (int)blockIdx.x - g.first_wg[ti], split = local / t.tiles_pad, pid = local - split * t.tiles_pad;
    if (pid >= t.tiles_n * g.tiles_m) return;   // padding: the whole workgroup leaves
    int tile_n, tile_m;
    tile_of_workgroup(t.tiles_n, g.tiles_m, pid, tile_n, tile_m);
    const int nb = g.nb, M = g.M;
    const int64_t K = (int64_t)nb * 256;
    const int n0 = tile_n * (32 * RW) + rg * 32, m0 = tile_m * TM;
    const int sb_begin = (int)((int64_t)nb * split / t.n_split), sb_end = (int)((int64_t)nb * (split + 1) / t.n_split);
    const int n_steps = (sb_end - sb_begin + KW - 1) / KW;

    S strip_src;
    {
        const int row0 = min(n0, t.N - 1);   // rows past the edge of the matrix repeat its last row (never stored)
        strip_src.init(t, nb, row0, min(t.N - 1 - row0, 31), lane);
    }
    uint8_t *strip = smem + L::kOffStrip + wave * S::kBytes;   // second buffer NW * kBytes further on
    auto my_sb = [&](int s) { return (uint32_t)min(sb_begin + s * KW + kp, sb_end - 1); };

    // activations: request p of a wave = K part p / AP, tokens 4*(wave + NW*(p % AP)) .. +3 of the tile
    constexpr int AP = 8 * JT / NW;
    const int mcap = min(M - 1 - m0, TM - 1);
    const int8_t *abase = scalar_pointer(g.qs + (int64_t)m0 * K);
    uint32_t aoff[AP];
#pragma unroll
    for (int j = 0; j < AP; ++j) {
        const int row = 4 * (wave + NW * j) + (lane >> 4), seg = (lane & 15) ^ (row & 15);
        aoff[j] = (uint32_t)(min(row, mcap) * (int)K + 16 * seg);
    }
    auto request_act = [&](int s, int p) {
        const uint32_t sb = (uint32_t)min(sb_begin + s * KW + p / AP, sb_end - 1);
        global_to_lds16(abase + (aoff[p % AP] + sb * 256u), smem + ((s & 1) * KW + p / AP) * L::kAct + (wave + NW * (p % AP)) * 1024);
    };
    auto request_acts = [&](int s) {
#pragma unroll
        for (int p = 0; p < KW * AP; ++p) request_act(s, p);
    };
    auto request_strip = [&](int s, uint8_t *dst) {
#pragma unroll
        for (int c = 0; c < S::kLoads; ++c) strip_src.request(my_sb(s), dst, c);
    };
    const uint8_t *msbase = nullptr;
    if constexpr (kQ4) {
        static_assert(KW * JT <= NW, "a wave requests one tile of the min-term plane at most");
        msbase = scalar_pointer(reinterpret_cast<const uint8_t *>(g.msum) + (int64_t)m0 * nb * 32);
    }
    // (three token tiles: worked out at every request from the lane counter.  Kept in a register it was spilled, and the wait
    // for its reload was one for everything outstanding; 4096 -> 40960 at 96 rows 66.6 -> 64.6 us.  Thirteen other registers of
    // that instance are spilled still, five of them since the arguments stand by field, and the step loop waits for their
    // reloads in the same way.  Calls of 1024 to 5120 weights a row at 65 to 96 rows are 0 to 3 % faster than before that.)
    auto ms_offset = [&]() {
        int zero = 0;
        if constexpr (JT >= 3) asm volatile("" : "+v"(zero));
        const int l = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, zero));
        return (uint32_t)(min((wave % JT) * 32 + (l >> 1), mcap) * nb * 32 + 16 * (l & 1));
    };
    auto request_ms = [&](int s) {
        if constexpr (kQ4) {
            if (wave < KW * JT) {
                const uint32_t sb = (uint32_t)min(sb_begin + s * KW + wave / JT, sb_end - 1);
                global_to_lds16(msbase + (ms_offset() + sb * 32u), smem + L::kOffMs + ((s & 1) * KW + wave / JT) * L::kMs + (wave % JT) * 1024);
            }
        }
    };
    // Scales go through LDS kScaleSb super-blocks at a time: a plain load in the loop below would make the compiler
    // wait for every outstanding request before its value is used.
    const global_ptr<float> dxbase = scalar_global(g.d + (int64_t)m0 * nb);
    float *const dx_lds = reinterpret_cast<float *>(smem + L::kOffDx);
    uint16_t *const dw_lds = reinterpret_cast<uint16_t *>(smem + L::kOffDw + wave * L::kDwWave);
    float rs_mine = 1.f;   // of token tid % TM
    float inv_rs = 1.f;
    if constexpr (kQ4) {   // the min-term operand is normalised by the row: see gemm_q4k_q8k_direct_kernel
        rs_mine = g.rs[m0 + min(tid % TM, mcap)];
        inv_rs = 1.0f / rs_mine;
    }
    auto load_scales = [&](int sb0) {
        // thread -> token tid % TM of super-blocks tid / TM, + NT / TM, ... (threads past the last whole group idle)
        constexpr int kGroups = NT / TM;
        if (tid < kGroups * TM) {
            const int tok = tid % TM;
#pragma unroll
            for (int i = 0; i < (L::kScaleSb + kGroups - 1) / kGroups; ++i) {
                const int q = tid / TM + i * kGroups;
                if (q < L::kScaleSb)
                    dx_lds[q * TM + tok] = load_global<float>(dxbase, 4u * (uint32_t)(min(tok, mcap) * nb + min(sb0 + q, sb_end - 1))) * inv_rs;
            }
        }
        if constexpr (!kQ4) {
#pragma unroll
            for (int i = 0; i < L::kScaleSb / KW / 2; ++i) {
                const int q = 2 * i + lh;   // the wave's q-th super-block of the chunk
                dw_lds[q * 32 + l32] = strip_src.scale((uint32_t)min(sb0 + q * KW + kp, sb_end - 1));
            }
        }
    };

    v16f acc[JT];
#pragma unroll
    for (int j = 0; j < JT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[j][v] = 0.f;
    const v16i zi = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const v16f zf = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // activation segment i + 8*(l/32) of token l%32 (+32*j) sits in slot (i + 8*(l/32)) ^ (l%16)
    const int aoffl = l32 * 256 + 16 * ((8 * lh) ^ (l32 & 15));

    constexpr int NC = JT < 4 ? JT : 1;   // token tiles whose chains are in registers at a time
    v16i ilo[NC], ihi[NC];
    float dn = 0.f;
    // the finished chains of tile j of step s into the accumulators
    auto flush_tile = [&](int j, int c, int s) {
        constexpr int kShift = kQ4 ? 3 : 8;
        const uint8_t *dxs = smem + L::kOffDx + ((s * KW) % L::kScaleSb + kp) * L::kDx;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // (as v4i: a float4 read here made the compiler wait for every outstanding request to LDS first)
            const v4i d4 = *reinterpret_cast<const v4i *>(dxs + (j * 32 + 8 * i + 4 * lh) * 4);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int v = 4 * i + r;
                acc[j][v] = fmaf((float)((ihi[c][v] << kShift) + ilo[c][v]), __int_as_float(d4[r]) * dn, acc[j][v]);
            }
        }
    };
    auto flush = [&](int s) {
        if constexpr (JT < 4) {
#pragma unroll
            for (int j = 0; j < JT; ++j) flush_tile(j, j, s);
        }
    };
    auto products = [&](const typename S::Raw &raw, bool live, int s, auto &&requests_of) {
        const uint8_t *ab = smem + ((s & 1) * KW + kp) * L::kAct;
        auto frag = [&](int j, int i) { return *reinterpret_cast<const v4i *>(ab + j * 8192 + (aoffl ^ (16 * i))); };
        v4i cl[8], ch[8];
        // the order in which the operands of the super-block's eight products come out of the raw block (Q6_K: a piece
        // of ql holds two of them)
        constexpr int kOrder[8] = {0, kQ4 ? 1 : 4, 2, kQ4 ? 3 : 6, kQ4 ? 4 : 1, 5, kQ4 ? 6 : 3, 7};
        uint32_t lo_w = 0, hi_w = 0;
        [[maybe_unused]] ScalesK4 sc;
        auto convert = [&](int p) {   // makes the operands of product kOrder[p] (Q6_K: at even p, of two)
            if constexpr (kQ4) {
                convert_q4k(raw.q[2 * (p >> 2) + (p & 1)], lo_w, hi_w, p >> 1, cl[p], ch[p]);
            } else if ((p & 1) == 0) {
                const int e = p >> 2, gl = (p >> 1) & 1;
                convert_q6k(raw.ql[2 * gl + e], raw.qh[e], raw.sc, gl, e, cl, ch);
            }
        };
        if constexpr (kQ4) {
            sc = unpack_scales_k4((uint32_t)raw.hdr[1], (uint32_t)raw.hdr[2], (uint32_t)raw.hdr[3]);
            dn = live ? h2f((uint32_t)raw.hdr[0] & 0xffffu) * kMinPrescale : 0.f;   // exact: a power of two
            const uint32_t scw = lh ? sc.sc_hi : sc.sc_lo;   // sub-blocks 4*(l/32) .. +3
            lo_w = scw & 0x07070707u;
            hi_w = (scw >> 3) & 0x07070707u;
        } else {
            dn = live ? h2f(dw_lds[(s * KW) % L::kScaleSb / KW * 32 + l32]) : 0.f;
        }
        // min term: the mins as exact fp16 integers against the plane's [high | low] halves, -dmin once per output
        [[maybe_unused]] v8h mins, am[JT];
        [[maybe_unused]] v16f msum[NC];
        [[maybe_unused]] float ndmin = 0.f;
        auto min_convert = [&]() {
            if constexpr (kQ4) {
                ndmin = live ? -h2f((uint32_t)raw.hdr[0] >> 16) : 0.f;
                mins = bytes_to_f16(sc.mn_lo, sc.mn_hi);
                const uint8_t *msb = smem + L::kOffMs + ((s & 1) * KW + kp) * L::kMs;
#pragma unroll
                for (int j = 0; j < JT; ++j) am[j] = *reinterpret_cast<const v8h *>(msb + (j * 32 + l32) * 32 + 16 * lh);
            }
        };
        auto min_multiply = [&](int j, int c) {
            if constexpr (kQ4) msum[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(am[j], mins, zf, 0, 0, 0);
        };
        auto min_add = [&](int j, int c) {
            if constexpr (kQ4) {
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[j][v] = fmaf(msum[c][v], ndmin, acc[j][v]);
            }
        };
        if constexpr (JT >= 4) {   // tile by tile: both chains of four tiles do not fit the registers
            static_assert(!kQ4, "Q4_K takes three token tiles at most");
#pragma unroll
            for (int p = 0; p < 8; ++p) convert(p);
        } else {
            // Pinned step by step: the activation fragments of two products are in flight, the next product's weights
            // are converted between the matrix instructions of this one.
            v4i af[3][JT];
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int j = 0; j < JT; ++j) af[p][j] = frag(j, kOrder[p]);
            convert(0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int p = 0; p < 8; ++p) {
                const int i = kOrder[p];
                if (p + 2 < 8) {
#pragma unroll
                    for (int j = 0; j < JT; ++j) af[(p + 2) % 3][j] = frag(j, kOrder[p + 2]);
                }
                if (p + 1 < 8 && (kQ4 || (p & 1))) convert(p + 1);
                requests_of(p);
                if (p == 2) min_convert();
#pragma unroll
                for (int j = 0; j < JT; ++j) {
                    ilo[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[p % 3][j], cl[i], p == 0 ? zi : ilo[j], 0, 0, 0);
                    ihi[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[p % 3][j], ch[i], p == 0 ? zi : ihi[j], 0, 0, 0);
                }
                if (p >= 3 && p < 3 + JT) min_multiply(p - 3, p - 3);
                if (p >= 4 && p < 4 + JT) min_add(p - 4, p - 4);
#pragma unroll
                for (int k = 0; k < 2 * JT; ++k) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (JT >= 4) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < JT; ++j) {
#pragma unroll
                for (int p = 0; p < 8; ++p) {
                    const int i = kOrder[p];
                    if (j == 0) requests_of(p);
                    const v4i a4 = frag(j, i);
                    ilo[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a4, cl[i], p == 0 ? zi : ilo[0], 0, 0, 0);
                    ihi[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a4, ch[i], p == 0 ? zi : ihi[0], 0, 0, 0);
                }
                flush_tile(j, 0, s);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    // ---- prologue: everything of step 0 and the strips of the steps the buffers hold
    request_strip(0, strip);
    request_acts(0);
    request_ms(0);
    load_scales(sb_begin);
    if constexpr (SW == 2) {
        request_strip(1, strip + NW * S::kBytes);
        wait_vmcnt<S::kLoads>();
    } else {
        wait_vmcnt<0>();
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // The two waves that share a SIMD (w and w + 4) work half a step apart: the EARLY ones (0..3) multiply, then flush;
    // the LATE ones flush the previous step first, so that one has vector work while the other has matrix work.
    auto run = [&](auto late_tag) {
        constexpr bool LATE = decltype(late_tag)::value && JT < 3;   // (no registers to spare beyond)
        // MORE1: another step follows; MORE2: so does one whose strip is requested now
        auto step = [&](int s, auto more1, auto more2) {
            constexpr bool MORE1 = decltype(more1)::value, MORE2 = decltype(more2)::value;
            uint8_t *sbuf = strip + (SW == 2 ? (s & 1) * NW * S::kBytes : 0);
            const typename S::Raw raw = S::read(sbuf, l32, lh);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the strip has been read: it may be overwritten
            // The step's requests, activations first, spread over its eight products: sent in one go they hold up all waves of the
            // workgroup at once (a compute unit takes 64 bytes of them a cycle).  14336 -> 4096 at 192 tokens 53.6 -> 48.8 us, gate +
            // up 4096 -> 2 x 14336 at 96 54.9 -> 51.0.  Q6_K in two K parts has its conversions to hide them: level to 2 % slower.
            constexpr bool kSpread = kQ4 || KW == 1;
            constexpr int kRequests = KW * AP + S::kLoads, kSlots = kSpread ? 8 : 1;
            auto requests_of = [&](int p) {
#pragma unroll
                for (int i = p * kRequests / kSlots; i < std::min((p + 1) * kRequests / kSlots, kRequests); ++i) {
                    if (i < KW * AP) {
                        if constexpr (MORE1) request_act(s + 1, i);
                    } else {
                        if constexpr (MORE2) strip_src.request(my_sb(s + SW), sbuf, i - KW * AP);
                    }
                }
            };
            if constexpr (MORE1) request_ms(s + 1);
            if constexpr (!kSpread) requests_of(0);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (LATE) {
                if (s > 0) flush(s - 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (s > 0 && (s * KW) % L::kScaleSb == 0) {   // the chunk of scales is used up
                __syncthreads();
                load_scales(sb_begin + s * KW);
                __syncthreads();
            }
            products(raw, sb_begin + s * KW + kp < sb_end, s, [&](int p) {
                if constexpr (kSpread) requests_of(p);
            });
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (!LATE) {
                flush(s);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (MORE1) {
                if constexpr (SW == 2 && MORE2) wait_vmcnt<S::kLoads>();   // all but the strip just asked for
                else wait_vmcnt<0>();
                // (__syncthreads would wait for every outstanding request)
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            }
        };
        int s = 0;
        for (; s + SW < n_steps; ++s) step(s, std::true_type{}, std::true_type{});
        if constexpr (SW == 2)
            for (; s + 1 < n_steps; ++s) step(s, std::true_type{}, std::false_type{});
        step(s, std::false_type{}, std::false_type{});
        if constexpr (LATE) flush(s);
    };
    if constexpr (NW <= 4) {   // a wave a SIMD
        run(std::false_type{});
    } else {
        if (wave < 4) run(std::false_type{});
        else run(std::true_type{});
    }

    // ---- the K parts meet in LDS: part q of a row group keeps token tiles j % KW == q, the others hand theirs over
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (a single step leaves its second strip request behind)
    float *const factor = reinterpret_cast<float *>(smem + L::kOffStrip);   // behind what the K parts exchange
    if constexpr (KW > 1 || kQ4) {
        __syncthreads();
        if (kQ4 && tid < TM) factor[tid] = rs_mine * (1.0f / kMinPrescale);   // the rows' factors (normaliser / 16)
        v4i *const meet = reinterpret_cast<v4i *>(smem);
        if constexpr (KW > 1) {
#pragma unroll
            for (int j = 0; j < JT; ++j)
                if (j % KW != kp) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        meet[((wave * JT + j) * 4 + i) * 64 + lane] =
                            v4i{__float_as_int(acc[j][4 * i]), __float_as_int(acc[j][4 * i + 1]), __float_as_int(acc[j][4 * i + 2]), __float_as_int(acc[j][4 * i + 3])};
                }
        }
        __syncthreads();
        if constexpr (KW > 1) {
#pragma unroll
            for (int j = 0; j < JT; ++j)
                if (j % KW == kp) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const v4i o = meet[(((kp ^ 1) * RW + rg) * JT + j) * 4 * 64 + i * 64 + lane];
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[j][4 * i + r] += __int_as_float(o[r]);   // two addends: either order
                    }
                }
        }
    }
    // ---- store: accumulator register v of lane l is token 8*(v/4) + 4*(l/32) + v%4, weight row l%32
    static_assert(KW <= 2, "more K parts than two have to be added in order");
    if (n0 + l32 >= t.N) return;
    float *const out = t.out + (size_t)split * ((size_t)M * t.N) + (size_t)m0 * t.N + n0;
    const int rows = M - m0;
#pragma unroll
    for (int j = 0; j < JT; ++j) {
        if (KW > 1 && j % KW != kp) continue;
        if (j * 32 >= rows) break;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v4i f4 = {0, 0, 0, 0};
            if constexpr (kQ4) f4 = *reinterpret_cast<const v4i *>(factor + j * 32 + 8 * i + 4 * lh);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = j * 32 + 8 * i + 4 * lh + r;
                const float v = kQ4 ? acc[j][4 * i + r] * __int_as_float(f4[r]) : acc[j][4 * i + r];
                if (m < rows) out[(uint32_t)(m * t.N + l32)] = v;
            }
        }
    }
}

// y_i = part_i[0] + part_i[1] + ... in that order, all matrices of a call in one launch
__global__ __launch_bounds__(256) void sum_parts_kernel(const SumTargets g) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    SumTarget t = g.t[0];
#pragma unroll
    for (int k = 1; k < kMaxTargets; ++k)
        if (k < g.n && (int64_t)blockIdx.x * 256 >= g.t[k].first) t = g.t[k];   // targets start at multiples of 256
    const int64_t e = i - t.first;
    if (e >= t.n4) return;
    const float4 *p = reinterpret_cast<const float4 *>(t.part) + e;
    float4 s = p[0];
    for (int c = 1; c < t.n_split; ++c) {
        const float4 v = p[(int64_t)c * t.n4];
        s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    reinterpret_cast<float4 *>(t.y)[e] = s;
}

struct StreamPlan {
    int jt, kw, n_split;
};
// token tiles a workgroup of the larger tile shape: as few as cover M in as few workgroups
int large_token_tiles(int64_t M) { return (int)std::max<int64_t>(2, ((M + 31) / 32 + (M + 127) / 128 - 1) / ((M + 127) / 128)); }
// workgroups of one stretch of K: tiles, filled up to the same number on each of the 8 XCDs
int64_t stream_tiles(int64_t M, int64_t N, int jt, int kw) {
    return ((N + 256 / kw - 1) / (256 / kw) * ((M + 32 * jt - 1) / (32 * jt)) + 7) / 8 * 8;
}

// One matrix's cut.  It depends on the matrix and the row count alone: a matrix is cut the same way whatever rides
// along with it, so the results of a call with several matrices are bit for bit those of separate calls.
StreamPlan stream_plan(int type, int64_t K, int64_t M, int64_t N) {
    StreamPlan p;
    const int64_t nb = K / 256, cus = cu_count();
    // Two K parts a workgroup (128 rows x 64 tokens) while that is one round of workgroups; beyond, 256 rows and as few
    // token tiles as cover M, so that a converted weight serves more tokens.
    const int large_jt = large_token_tiles(M);
    const int64_t small_tiles = stream_tiles(M, N, 2, 2);
    bool large = small_tiles > cus;
    // Q6_K conversions are dear: beyond 128 tokens long rows take the larger tile as well (14336 -> 4096 at 192 tokens 53.5 us
    // in 64-token tiles, 44.1 in 96-token ones, 28672 -> 8192 186.5 against 133.7), unless that means twelve and more
    // stretches: their partial tiles cost more than they bring (8192 -> 1024 at 160 / 250 tokens 25.3 / 28.6 us, in 64-token tiles
    // 22.8 / 24.3; 8192 -> 2048 29.1 / 33.3 and 27.5 / 29.3) and lengthen the sums (14336 -> 1024 against 64 bits 1.07e-7 and 8.0e-8).
    if (type == kTypeQ6_K && M > 128 && K >= 8192)
        large = large || !(N > 512 && K <= 16384 && stream_tiles(M, N, large_jt, 1) * 12 <= cus);
    p.jt = large ? large_jt : 2;
    p.kw = large ? 1 : 2;
    p.jt = tuning_int("QPROJ_STREAM_JT", p.jt);
    p.kw = tuning_int("QPROJ_STREAM_KW", p.kw);
    // Stretches of K over workgroups, by what usually shares the launch (a matrix has to be cut without knowing it, and
    // launch_group evens out the workgroups where the guess leaves half the chip idle): a matrix with N > K has a sibling of its size
    // (gate / up) and takes half the chip, a square one (q, o) leaves room for k and v, a down projection or a matrix of
    // long rows takes all of it.  Measured, us, 160 / 256 workgroups: q/k/v of 4096 at 96 tokens 21.5 / 25.6, o 17.4 / 15.9;
    // gate + up 4096 -> 14336 at 64 tokens 27.3 / 38.3; 14336 -> 4096 39.0 / 26.3 at 96 tokens; 8192 x 8192 40.1 / 28.3.
    // (Rows of 8192 and more stay cut beside a sibling of their size too: 8192 -> 2 x 28672 at 80 tokens takes 154 us in two
    // stretches each and 139 whole, 182 in the tiled kernels, but whole its sums run over 32 super-blocks instead of 16.)
    const bool whole_chip = K > N || K >= 8192 || (K == N && type == kTypeQ6_K);
    const int64_t wgs = tuning_int("QPROJ_STREAM_WGS", whole_chip ? (int)cus : (int)(K == N ? cus * 5 / 8 : cus / 2));
    int64_t n = std::max<int64_t>(1, wgs / stream_tiles(M, N, p.jt, p.kw));
    // Beyond 256 tokens k and v stay whole where q and they are one round together, or nearly one and a half: cut, they cost the
    // adding pass and more starts than they fill (q/k/v of 3072 at 384 tokens 37.4 -> 26.6 us, of 4096 at 512 56.8 -> 52.3, of 2048
    // at 640 29.5 -> 22.4; 1.1 rounds, 4096 at 384 tokens, 46.0 cut and 50.1 whole).  In a call of its own a small one is the
    // slower for it: 4096 -> 256 / 512 / 1024 at 288 tokens 19.6 us in the 64-token tiles, cut in stretches, and 22.0 whole here, 20.3 / 22.2,
    // 22.3 / 22.5; 5120 -> 512 at 288 21.8 / 26.0; 4096 -> 1024 at 512 24.6 / 23.9.
    if (M > 256 && N <= 1024 && K > N) {
        const int64_t together = stream_tiles(M, K, p.jt, p.kw) + 2 * stream_tiles(M, N, p.jt, p.kw);
        if (together <= cus || together * 5 >= cus * 7) n = 1;
    }
    n = tuning_int("QPROJ_STREAM_SPLIT", (int)n);
    n = std::min<int64_t>(n, std::max<int64_t>(1, nb / (2 * p.kw)));   // two steps a stretch at least
    // never more partial tiles than the allocation-free entry point has room for beside the activation planes
    n = std::min<int64_t>(n, std::max<int64_t>(1, (int64_t)(q8k_scratch_room(M, K) / ((size_t)M * N * 4))));
    // (a cut in two of short rows leaves no room for k and v in the round: 2560 -> 2560 / 1024 / 1024 at 250 tokens 34.9 -> 25.5
    // us with it whole, 3072 -> 3072 / 1024 / 1024 at 192 31.0 -> 27.9)
    if (K == N && n == 2 && nb < 14 && stream_tiles(M, N, p.jt, p.kw) * 4 > cus) n = 1;
    const auto steps = [&](int64_t parts) { return ((nb + parts - 1) / parts + p.kw - 1) / p.kw; };
    while (n > 1 && steps(n - 1) == steps(n)) --n;   // no more stretches than it takes
    if ((M * N) % 4 != 0) n = 1;
    p.n_split = (int)n;
    return p;
}

template <int QT, int JT, int KW, int SW, int NW>
hipError_t launch_stream_kernel(const StreamArgs &g, int wgs, hipStream_t s) {
    constexpr int lds = StreamLds<QT, JT, KW, SW, NW>::kTotal;
    const auto kern = &gemm_stream_kernel<QT, JT, KW, SW, NW>;
    static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(64 * NW), lds, s, g);
    return hipGetLastError();
}

using LaunchFn = hipError_t (*)(const StreamArgs &, int, hipStream_t);
LaunchFn instance(int type, int jt, int kw, int waves) {   // null: not built
#define QP_STREAM(QT, JT, KW, SW, NW) \
    if (type == QT && jt == JT && kw == KW && waves == NW) return &launch_stream_kernel<QT, JT, KW, SW, NW>
    // (64-token tiles with K in one part are only taken by grids beyond a round of the halves)
    QP_STREAM(kTypeQ4_K, 2, 1, 2, 8);
    QP_STREAM(kTypeQ4_K, 2, 2, 2, 8);
    QP_STREAM(kTypeQ4_K, 2, 2, 2, 4);
    QP_STREAM(kTypeQ4_K, 3, 1, 2, 8);
    QP_STREAM(kTypeQ4_K, 3, 1, 2, 4);
    QP_STREAM(kTypeQ6_K, 2, 1, 2, 8);
    QP_STREAM(kTypeQ6_K, 2, 2, 1, 8);
    QP_STREAM(kTypeQ6_K, 2, 2, 1, 4);
    QP_STREAM(kTypeQ6_K, 3, 1, 1, 8);
    QP_STREAM(kTypeQ6_K, 3, 1, 1, 4);
    QP_STREAM(kTypeQ6_K, 4, 1, 1, 8);
    QP_STREAM(kTypeQ6_K, 4, 1, 1, 4);
#undef QP_STREAM
    return nullptr;
}

}  // namespace

// Which products the streaming kernel takes.  From 33 tokens (below, the small-batch kernel) to 256, and Q4_K beyond while its
// 64-token tiles are one round of workgroups: square and narrow matrices, which the 64-token tiles of
// gemm_q4k_q8k_direct_kernel walk a super-block at a time with one in flight.  us a call, there / here: 4096 x 4096 at 257 / 384 / 512
// tokens 34.5 / 27.9, 36.7 / 29.7, 40.1 / 32.5; 3072 x 3072 at 320 29.1 / 19.5; 2048 x 2048 at 1024 27.0 / 23.2; 8192 -> 3072 at 448 75.3 /
// 46.7; 4096 -> 1024 at 1536 40.6 / 32.9; q/k/v of 4096 at 320 / 384 / 512 65.8 / 31.6, 53.0 / 46.1, 56.3 / 52.9, of 2048 at 512 39.4 / 20.1, at
// 1024 35.7 / 35.0.  k and v follow q: streamed without it, 4096 -> 4096 / 1024 / 1024 at 640 tokens 58.9 / 86.  (Q6_K would gain as much,
// 3072 q/k/v at 320 tokens 61.8 / 32.8, but with sums 1 to 4 % further from 64 bits than the stretches of its 64-token tiles.)
// Left slower: q/k/v of fewer than 2048 weights a row where the three are more than one round together, which a matrix does not
// know of: three of 1280 at 576 / 1024 tokens 25.2 / 28.7, 29.1 / 32.3, 1536 with 1024 for k and v at 768 28.5 / 29.6; the same square matrix alone (o) gains at those
// sizes, 1280 at 1024 19.9 / 18.8.  Four waves a workgroup there are slower still.
// Of the grids beyond one round of workgroups Q4_K keeps the older tiles from 97 tokens on, where arithmetic and not latency is the limit
// (4096 -> 32000 at 128 tokens 51.0 us there, 54.0 here; at 96 tokens 50.1 against 45.3).  The 128-token kernels
// keep the grids they fill (q4k_fills_wide, q6k_fills_wide) where they are as fast or faster, us there / here: Q4_K beyond
// 128 tokens (28672 -> 8192 at 192 / 256 tokens 147 / 159, 151 / 166) and from 65 on for very long rows (28672 -> 16384 at 112
// tokens 155 / 165); Q6_K where the tokens fill 128-token tiles (8192 -> 2 x 28672 at 256 tokens 334 / 346, 4096 -> 32000
// 91.5 / 96.1) and from 65 on for long rows (12288 x 12288 at 96 tokens 79 / 88, 16384 x 16384 109 / 124).  At 129..192 tokens
// Q6_K has tiles of 96 here: 4096 -> 32000 at 160 tokens 91.7 / 83.
bool stream_takes(int type, int64_t K, int64_t M, int64_t N) {
    const int lo = tuning_int("QPROJ_STREAM_MIN_M", 33), hi = tuning_int("QPROJ_STREAM_MAX_M", type == kTypeQ4_K ? 2048 : 256);
    if ((type != kTypeQ4_K && type != kTypeQ6_K) || K % 256 != 0 || K > (1 << 22) || M < lo || M > hi) return false;
    if (N > (1 << 24)) return false;   // row and tile numbers are ints, a tile's outputs are indexed with 32 bits: 127 * N + 31 at most
    if (type == kTypeQ6_K) {
        const int jt = large_token_tiles(M);
        // half a round of 128-token tiles and, with more than four times K rows (an output head), nothing that rides along
        const bool alone = M <= 128 && jt == 4 && N > 4 * K && stream_tiles(M, N, 4, 1) * 2 <= cu_count() && stream_tiles(M, N, 2, 2) > cu_count();
        return !alone && !((jt == 4 || (jt == 3 && M <= 96 && K >= 12288)) && q6k_fills_wide(K, M, N));
    }
    if ((M > 128 || (M > 64 && K >= 16384)) && q4k_fills_wide(K, M, N)) return false;
    if (M <= 96) return true;
    if (M > 256 && N <= 1024 && stream_tiles(M, K, 2, 2) > cu_count()) return false;   // k and v go with q
    // (beyond 256 tokens up rides along with gate: 1024 -> 2 x 4096 at 320 tokens 21.2 / 22.7)
    return stream_tiles(M, N, 2, 2) * (M > 256 && N > K ? 2 : 1) <= cu_count();
}

namespace {
size_t partial_bytes(const StreamPlan &p, int64_t M, int64_t N) { return p.n_split > 1 ? (size_t)p.n_split * M * N * 4 : 0; }

// How many of the matrices from `first` on have room for their partial tiles in `bytes` of scratch; the next ones follow
// in launches of their own, behind the adding pass, through the same bytes.
int matrices_that_fit(int n, const StreamPlan *plans, int64_t M, const int64_t *N, int first, size_t bytes, size_t *used) {
    *used = 0;
    int i = first;
    for (; i < n; ++i) {
        const size_t b = partial_bytes(plans[i], M, N[i]);
        if (*used + b > bytes) break;
        *used += b;
    }
    return i - first;
}
}  // namespace

// Scratch for the matrices of one call: all partial tiles side by side where the allocation-free entry point has the
// room, else the largest run of matrices that has it (8192 -> 8192 / 1024 / 1024, Q6_K, 256 rows: 33.5 + 16.8 + 16.8 MB)
size_t stream_scratch_bytes(int type, int64_t K, int64_t M, int n, const int64_t *N) {
    StreamPlan plans[kMaxTargets];
    for (int i = 0; i < n; ++i) plans[i] = stream_plan(type, K, M, N[i]);
    size_t need = 0;
    for (int first = 0; first < n;) {
        size_t used = 0;
        first += std::max(1, matrices_that_fit(n, plans, M, N, first, q8k_scratch_room(M, K), &used));   // (alone each fits: stream_plan)
        need = std::max(need, used);
    }
    return need;
}

namespace {
// the matrices of one launch group, their partial tiles side by side in `part`: a launch for all of one tile shape
// (q/k/v, gate/up: all of them), then one adding pass
hipError_t launch_group(int n, const WeightView *w, const StreamPlan *plans, const ActView &a, int64_t M, float *const *y, float *part, hipStream_t s) {
    const bool q4 = w[0].type == kTypeQ4_K;
    SumTargets sg{};
    float *out[kMaxTargets];
    for (int i = 0; i < n; ++i) {
        out[i] = y[i];
        if (plans[i].n_split == 1) continue;
        if (!dry_run()) {
            out[i] = part;
            part += partial_bytes(plans[i], M, w[i].N) / 4;
        }
        add_sum(sg, out[i], y[i], plans[i].n_split, M * w[i].N);
    }
    if (sg.n && dry_run()) plan_note_cut();
    bool done[kMaxTargets] = {};
    for (int first = 0; first < n; ++first) {
        if (done[first]) continue;
        const StreamPlan &p0 = plans[first];
        StreamArgs g{};
        int count = 0;
        for (int i = 0; i < kMaxTargets; ++i) g.first_wg[i] = INT_MAX;
        g.qs = a.qs;
        g.d = a.d;
        g.msum = a.msum;
        g.rs = a.rs;
        g.M = (int)M;
        g.nb = (int)(w[0].K / 256);
        g.tiles_m = (int)((M + 32 * p0.jt - 1) / (32 * p0.jt));
        const auto tiles_pad = [&](int i, int rows) { return ((w[i].N + rows - 1) / rows * g.tiles_m + 7) / 8 * 8; };
        // Four waves a workgroup (half the weight rows) where that many workgroups are still one round: the same sums, on
        // twice the compute units.  Eight waves -> four, us a call: Q4_K 4096 -> 14336 alone at 48 rows 27.8 -> 23.3, 4096 x
        // 4096 18.4 -> 16.6; Q6_K 4096 -> 14336 33.5 -> 27.8 at 48 rows, 69.3 -> 52.0 at 160; Q4_K 4096 -> 32000 at 96 rows
        // 69.6 -> 50.8.  (A matrix is cut as if its usual neighbours rode along; alone it left half the chip idle.)
        int64_t halves = 0;
        for (int i = first; i < n; ++i)
            if (plans[i].jt == p0.jt && plans[i].kw == p0.kw) halves += tiles_pad(i, 128 / p0.kw) * plans[i].n_split;
        const int waves = tuning_int("QPROJ_STREAM_WAVES", halves <= cu_count() ? 4 : 8), rows = 32 * waves / p0.kw;
        int64_t wg = 0;
        for (int i = first; i < n; ++i) {
            if (plans[i].jt != p0.jt || plans[i].kw != p0.kw) continue;
            done[i] = true;
            const int c = count++;
            if (q4) g.p0[c] = w[i].q4k;
            else {
                g.p0[c] = w[i].q6_ql;
                g.p1[c] = w[i].q6_qh;
                g.p2[c] = reinterpret_cast<const uint8_t *>(w[i].q6_sc);
                g.p3[c] = reinterpret_cast<const uint8_t *>(w[i].q6_d);
            }
            g.N[c] = (int)w[i].N;
            g.tiles_n[c] = (int)((w[i].N + rows - 1) / rows);
            g.tiles_pad[c] = (int)tiles_pad(i, rows);
            g.n_split[c] = plans[i].n_split;
            g.first_wg[c] = (int)wg;
            g.out[c] = out[i];
            wg += (int64_t)g.tiles_pad[c] * g.n_split[c];
            plan_note("gemm_stream_kernel<%s, %d token tiles, %d K parts>%s: tile %d tokens x %d rows, %d tiles x %d K stretches%s", plan_type_name(w[0].type),
                      p0.jt, p0.kw, count > 1 ? " (same launch)" : "", 32 * p0.jt, rows, g.tiles_n[c] * g.tiles_m, g.n_split[c],
                      g.n_split[c] > 1 ? " + sum_parts_kernel" : "");
        }
        if (wg >= 0x7fffffff) return hipErrorInvalidValue;
        const LaunchFn run = instance(w[0].type, p0.jt, p0.kw, waves);
        if (!run) return hipErrorInvalidValue;   // (in a dry run too)
        if (dry_run()) continue;
        const hipError_t e = run(g, (int)wg, s);
        if (e != hipSuccess) return e;
    }
    if (dry_run() || sg.n == 0) return hipSuccess;
    return launch_sum_parts(sg, s);
}
}  // namespace

// n matrices of one type over the same activation rows; `scratch`: stream_scratch_bytes
hipError_t launch_gemm_stream(int n, const WeightView *w, const ActView &a, int64_t M, float *const *y, const Scratch &scratch,
                              hipStream_t s) {
    if (n < 1 || n > kMaxTargets || a.kind != kActKindQ8_K || M <= 0) return hipErrorInvalidValue;
    if (w[0].type == kTypeQ4_K && (!a.msum || !a.rs)) return hipErrorInvalidValue;
    StreamPlan plans[kMaxTargets];
    int64_t N[kMaxTargets];
    for (int i = 0; i < n; ++i) {
        if (w[i].type != w[0].type || w[i].K != w[0].K || !stream_takes(w[i].type, w[i].K, M, w[i].N)) return hipErrorInvalidValue;
        plans[i] = stream_plan(w[i].type, w[i].K, M, w[i].N);
        N[i] = w[i].N;
    }
    for (int first = 0; first < n;) {
        size_t used = 0;
        const int count = matrices_that_fit(n, plans, M, N, first, scratch.bytes, &used);
        if (count == 0 || (used && !scratch.p && !dry_run())) return hipErrorInvalidValue;   // partial tiles would not fit
        const hipError_t e = launch_group(count, w + first, plans + first, a, M, y + first, scratch.p, s);
        if (e != hipSuccess) return e;
        first += count;
    }
    return hipSuccess;
}

hipError_t launch_sum_parts(const SumTargets &g, hipStream_t s) {
    hipLaunchKernelGGL(sum_parts_kernel, dim3((unsigned)(g.threads / 256)), dim3(256), 0, s, g);
    return hipGetLastError();
}

}  // namespace qproj
