// Decode-regime projection (1..4 activation rows): a persistent, software-pipelined GEMV.
//
// One 1024-thread workgroup per CU.  The workgroup quantizes the activation rows (or copies
// rows quantized earlier) into LDS once; when a single K-chunk covers the whole row every lane
// then keeps its slice of the activations in registers for the rest of the kernel.  Each of
// the 16 waves walks its own run of consecutive weight rows, R at a time, with two register
// buffers filled and drained alternately, so the loads of step i+1 are outstanding while step i
// is computed.  Row addresses are a wave-uniform base plus 32-bit offsets, so the scalar unit
// does a handful of operations per step and the vector unit only the dot products.
#include "actquant_device.h"
#include "gemv_frags.h"
#include <limits.h>
#include <stddef.h>
#include <stdio.h>

namespace qproj {

namespace {

constexpr int kDecodeThreads = 1024;
constexpr int kDecodeWaves = kDecodeThreads / 64;

// Arguments of a launch.  A workgroup begins with a chain of trips to memory (arguments, activation row, weights), and
// arguments come a 64-byte line at a time: what every workgroup needs first are the kernel's leading parameters, what it
// needs of its matrix stands by field, so that Q4_K touches three lines and asks for them at once.  Before, 616 bytes loaded
// where they were used, us a launch: 4096 -> 4096 / 1024 / 1024 and 4096 x 4096 Q4_K 6.3 -> 5.7, Q6_K 14336 -> 4096 12.0 -> 11.5, Q8_0
// 2048 x 2048 4.1 -> 3.9.  (All ten lines asked for at once: 4 % slower than before.  The leading parameters preloaded into
// scalar registers by the dispatcher: level.)
struct DecodeArgs {
    int first_wave[kMaxTargets];       // of each matrix, counted over the launch; INT_MAX where there is none
    int rows_per_pair[kMaxTargets];    // consecutive rows each pair of neighbouring waves walks
    int64_t N[kMaxTargets];
    float *y[kMaxTargets];
    const uint8_t *p0[kMaxTargets];    // Q4_K: blocks; Q6_K: ql, qh, scales, d; Q8_0: quants, d
    const uint8_t *p1[kMaxTargets], *p2[kMaxTargets], *p3[kMaxTargets];
    const int8_t *qs;                  // rows quantized earlier
    const float *d;
    const int16_t *bsums;
};

template <int QT>
__device__ __forceinline__ WeightView weight_view(const DecodeArgs &args, int i, int64_t K, int nb) {
    WeightView w{};
    w.K = K;
    w.nb = nb;
    w.N = args.N[i];
    if constexpr (QT == kTypeQ4_K) {
        w.q4k = args.p0[i];
    } else if constexpr (QT == kTypeQ6_K) {
        w.q6_ql = args.p0[i];
        w.q6_qh = args.p1[i];
        w.q6_sc = reinterpret_cast<const int8_t *>(args.p2[i]);
        w.q6_d = reinterpret_cast<const uint16_t *>(args.p3[i]);
    } else {
        w.q8_qs = reinterpret_cast<const int8_t *>(args.p0[i]);
        w.q8_d = reinterpret_cast<const uint16_t *>(args.p1[i]);
    }
    return w;
}

// activations into LDS: FUSE quantizes fp32 rows here; otherwise planes quantized earlier are copied
// 256-wide pieces of an activation row that a wave fetches ahead of its first weights: four a row for one or two
// rows (K up to 16384 is covered; pieces fetched inside the quantizing loop instead come one after the other, a trip to
// L2 each: the down projection at two rows, 3.5 pieces a row and wave, 20.2 -> 17.5 us with one-row steps, then
// this), one a row for four rows (which take this kernel for K <= 4096 only)
__host__ __device__ constexpr int prefetched_pieces(int mt) { return mt <= 2 ? 4 : 1; }

template <int QT, int MT, bool FUSE>
__device__ __forceinline__ void stage_activations(uint8_t *smem, const DecodeArgs &args, const float *rows, int M, int64_t K, int kpad,
                                                  const float4 *first = nullptr) {
    constexpr int BLK = Geo<QT>::kBlk;
    int8_t *sq = reinterpret_cast<int8_t *>(smem);
    float *sd = reinterpret_cast<float *>(smem + MT * kpad);
    int16_t *sb = reinterpret_cast<int16_t *>(smem + MT * kpad + MT * (kpad / BLK) * 4);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int m = 0; m < MT; ++m) {
        const bool have = m < M;
        if (FUSE) {
            const float *x = rows + (int64_t)m * K;
            const int n_chunks = (int)((K + 255) / 256);
            for (int ch = wave; ch < n_chunks; ch += kDecodeWaves) {
                const int e0 = ch * 256 + 4 * lane;
                float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
                constexpr int kPer = prefetched_pieces(MT);   // pieces per row the caller fetched
                if (first && ch < wave + kDecodeWaves * kPer)
                    v = first[m * kPer + (ch - wave) / kDecodeWaves];
                else if (have && e0 < K) v = *reinterpret_cast<const float4 *>(x + e0);
                if (is_q8_0<QT>) {
                    int s;
                    float dd;
                    const uint32_t packed = wave_quantize_q8_32(v, s, dd);
                    if (e0 < K) {
                        *reinterpret_cast<uint32_t *>(sq + m * kpad + e0) = packed;
                        if ((lane & 7) == 0) sd[m * (kpad / 32) + (e0 >> 5)] = h2f(f2h(dd));
                    }
                } else {
                    int bsum;
                    float dd;
                    const uint32_t packed = wave_quantize_q8k(v, lane, bsum, dd);
                    *reinterpret_cast<uint32_t *>(sq + m * kpad + e0) = packed;
                    if ((lane & 3) == 0) sb[m * (kpad / 16) + ch * 16 + (lane >> 2)] = (int16_t)bsum;
                    if (lane == 0) sd[m * (kpad / 256) + ch] = dd;
                }
            }
        } else {
            const DecodeArgs &a = args;
            for (int i = tid; i < K / 16; i += kDecodeThreads) {
                uint4 v = make_uint4(0, 0, 0, 0);
                if (have) v = *reinterpret_cast<const uint4 *>(a.qs + (int64_t)m * K + i * 16);
                *reinterpret_cast<uint4 *>(sq + m * kpad + i * 16) = v;
            }
            for (int i = tid; i < K / BLK; i += kDecodeThreads)
                sd[m * (kpad / BLK) + i] = have ? a.d[(int64_t)m * (K / BLK) + i] : 0.f;
            if (!is_q8_0<QT>)
                for (int i = tid; i < K / 16; i += kDecodeThreads)
                    sb[m * (kpad / 16) + i] = have ? a.bsums[(int64_t)m * (K / 16) + i] : (int16_t)0;
        }
    }
}

template <int QT, int R>
__device__ __forceinline__ void issue(Raw<QT> (&raw)[R], const RowPtr<QT> &rp, int g, int c, int last_row, int nb, int lane) {
    constexpr int BPC = Geo<QT>::kChunk / Geo<QT>::kBlk;
    // Lanes past the end of a row (last, partial chunk) and rows past the end of the run load the
    // last valid block / row instead: always in bounds, never used.
    int blk = c * BPC + lane / Geo<QT>::kLanesPerBlk;
    if (blk >= nb) blk = nb - 1;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int rel = g * R + r;
        if (rel > last_row) rel = last_row;
        raw[r].load(rp, (uint32_t)blk, lane, (uint32_t)rel);
    }
}

// gate / up pairing: step g is row g of both tensors
template <int QT>
__device__ __forceinline__ void issue_pair(Raw<QT> (&raw)[2], const RowPtr<QT> &rp_gate, const RowPtr<QT> &rp_up, int g, int c,
                                           int last_row, int nb, int lane) {
    constexpr int BPC = Geo<QT>::kChunk / Geo<QT>::kBlk;
    int blk = c * BPC + lane / Geo<QT>::kLanesPerBlk;
    if (blk >= nb) blk = nb - 1;
    const int rel = g > last_row ? last_row : g;
    raw[0].load(rp_gate, (uint32_t)blk, lane, (uint32_t)rel);
    raw[1].load(rp_up, (uint32_t)blk, lane, (uint32_t)rel);
}

// XREG: the lane's activation slices live in `xr` (one chunk covers K); otherwise they are read
// from the LDS image for chunk c.  PAIR (R = 2): the two rows of a step are row g of the gate and of the up
// tensor, and what is stored is silu(gate) * up.
template <int QT, int MT, int R, bool XREG, bool PAIR = false>
__device__ __forceinline__ void consume(const Raw<QT> (&raw)[R], float (&acc)[MT][R], const Dot<QT> (&xr)[MT], const XTile &xt,
                                        int g, int c, int nch, int nb, int n_rows, int64_t row_begin, int64_t N,
                                        float *y, int M, int lane) {
    constexpr int CH = Geo<QT>::kChunk;
    if (lane_block<QT>((int64_t)c * CH, lane) < nb) {
        Frag<QT> f[R];
#pragma unroll
        for (int r = 0; r < R; ++r) f[r].unpack(raw[r], lane);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            if (XREG) {
#pragma unroll
                for (int r = 0; r < R; ++r) acc[m][r] += xr[m].dot(f[r]);
            } else {
                Dot<QT> dx;
                dx.load_x(xt, m, c * CH, lane);
#pragma unroll
                for (int r = 0; r < R; ++r) acc[m][r] += dx.dot(f[r]);
            }
        }
    }
    if (c + 1 == nch) {  // row group finished: reduce over the wave, store, start over
        constexpr int V = MT * R;
#pragma unroll
        for (int v0 = 0; v0 < V; v0 += 4) {
            float q[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) q[i] = (v0 + i < V) ? acc[(v0 + i) / R][(v0 + i) % R] : 0.f;
            const float t = wave_sum4(q, lane);
            const int i = lane - 12;  // lanes 12..15 hold the four sums
            if constexpr (PAIR) {
                const float up = dpp_move<0x101>(t);   // row_shl:1: sums 2m (gate) and 2m+1 (up) sit in neighbouring lanes
                if (i >= 0 && i < 4 && v0 + i < V && ((v0 + i) & 1) == 0) {
                    const int m = (v0 + i) / 2;
                    if (m < M && g < n_rows) y[(int64_t)m * N + row_begin + g] = (t / (1.0f + expf(-t))) * up;
                }
            } else if (i >= 0 && i < 4 && v0 + i < V) {
                const int m = (v0 + i) / R, r = (v0 + i) % R;
                if (m < M && g * R + r < n_rows) y[(int64_t)m * N + row_begin + g * R + r] = t;
            }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int r = 0; r < R; ++r) acc[m][r] = 0.f;
    }
}

template <int QT, int MT, int R, bool XREG, bool FUSE, bool PAIR = false>
__global__ __launch_bounds__(kDecodeThreads) void gemv_decode_kernel(const float *x, const float *norm_gamma, int K32, int nb, int kpad, int M,
                                                                     float norm_eps, int norm, const DecodeArgs args) {
    static_assert(!PAIR || R == 2, "the gate/up pairing walks two rows a step");
    extern __shared__ __align__(16) uint8_t smem[];
    constexpr int kPointers = QT == kTypeQ4_K ? 1 : is_q8_0<QT> ? 2 : 4;
    using Kernel = decltype(gemv_decode_kernel<QT, MT, R, XREG, FUSE, PAIR>);
    static_assert(offsetof(DecodeArgs, p3) == offsetof(DecodeArgs, p0) + 3 * sizeof(DecodeArgs::p0), "a format's pointers stand together");
    fetch_arguments<Kernel, argument_block(static_cast<Kernel *>(nullptr)).last + offsetof(DecodeArgs, p0) + kPointers * sizeof(DecodeArgs::p0)>();
    constexpr int CH = Geo<QT>::kChunk;
    constexpr int BLK = Geo<QT>::kBlk;
    const int lane = threadIdx.x & 63;
    const int wave = uniform(threadIdx.x >> 6);
    const int gw = blockIdx.x * kDecodeWaves + wave;  // global wave index
    const int64_t K = K32;
    const int nch = XREG ? 1 : kpad / CH;

    // The wave's piece of the activation row is requested BEFORE the first weights: loads return in order, and
    // behind a step of weights coming from HBM the quantizing prologue would wait two microseconds for sixteen
    // bytes that sit in L2 (phase clocks: staging 3000-4400 cycles of a workgroup's 25000).
    float4 x_first[MT * prefetched_pieces(MT)];
    if (FUSE) {
        constexpr int kPer = prefetched_pieces(MT);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                const int e0 = (wave + kDecodeWaves * i) * 256 + 4 * lane;
                x_first[m * kPer + i] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (m < M && e0 < K) x_first[m * kPer + i] = *reinterpret_cast<const float4 *>(x + (int64_t)m * K + e0);
            }
    }
    // RMS norm fused in front of the quantizer (the launcher only asks for it when the prefetched pieces are the
    // whole row): weights of the norm fetched with the row, sum of squares over the workgroup in the order of
    // the standalone kernel, then the pieces are replaced by (x * scale) * gamma.
    float4 g_first[prefetched_pieces(MT)];
    if (FUSE && norm) {
#pragma unroll
        for (int i = 0; i < prefetched_pieces(MT); ++i) {
            const int e0 = (wave + kDecodeWaves * i) * 256 + 4 * lane;
            g_first[i] = make_float4(1.f, 1.f, 1.f, 1.f);
            if (norm_gamma && e0 < K) g_first[i] = *reinterpret_cast<const float4 *>(norm_gamma + e0);
        }
    }

    // this wave's target and run of rows (selected once; everything below is wave-uniform)
    int ti = 0;
#pragma unroll
    for (int i = 1; i < kMaxTargets; ++i)
        if (!PAIR && gw >= args.first_wave[i]) ti = i;
    const WeightView w = weight_view<QT>(args, ti, K, nb);
    float *const y = args.y[ti];
    const int wave_first = args.first_wave[ti], rpp = args.rows_per_pair[ti];
    const int64_t N = w.N;
    // Rows are dealt to pairs of neighbouring waves: rpp consecutive rows a pair, the even wave taking the larger
    // part.  A target with 1.5 rows per wave then keeps every wave busy (2 + 1) where whole rows per wave would
    // leave a third of the workgroups without work, and with two rows a step the even wave's part is rounded up
    // to an even count so that no step fetches its last row twice (7 + 7 becomes 8 + 6).
    const int wl = gw - wave_first;
    int part_even = (rpp + 1) >> 1;
    if (!PAIR && R == 2) part_even = (part_even + 1) & ~1;
    if (part_even > rpp) part_even = rpp;
    const int64_t row_begin = (int64_t)(wl >> 1) * rpp + ((wl & 1) ? part_even : 0);
    const int own = (wl & 1) ? rpp - part_even : part_even;
    int n_rows = 0;  // rows this wave owns
    if (row_begin < N) n_rows = (int)((N - row_begin) < own ? (N - row_begin) : own);
    n_rows = uniform(n_rows);
    const int n_groups = PAIR ? n_rows : (n_rows + R - 1) / R;
    const int n_iter = n_groups * nch;
    const int last_row = n_rows > 0 ? n_rows - 1 : 0;
    RowPtr<QT> rp, rp_up;
    rp.set(w, row_begin < N ? row_begin : 0);
    rp_up.set(PAIR ? weight_view<QT>(args, 1, K, nb) : w, row_begin < N ? row_begin : 0);
    auto issue_rows = [&](Raw<QT> (&raw)[R], int g, int c) {
        if constexpr (PAIR) issue_pair<QT>(raw, rp, rp_up, g, c, last_row, nb, lane);
        else issue<QT, R>(raw, rp, g, c, last_row, nb, lane);
    };

    Raw<QT> buf_a[R], buf_b[R];
    issue_rows(buf_a, 0, 0);  // in flight while the activations are staged
    if (FUSE && norm) {
        __shared__ double norm_partial[kDecodeWaves];
        constexpr int kPer = prefetched_pieces(MT);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            double sq = 0.0;
#pragma unroll
            for (int i = 0; i < kPer; ++i) sq += sum4_sq(x_first[m * kPer + i]);
            if (m > 0) __syncthreads();   // the partial sums of the previous row have been read
            const double total = workgroup_sum16(sq, norm_partial);
            const float mean = (float)(total / (double)K);
            const float scale = 1.0f / sqrtf(mean + norm_eps);
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                float4 &v = x_first[m * kPer + i];
                v.x *= scale; v.y *= scale; v.z *= scale; v.w *= scale;
                if (norm_gamma) {
                    v.x *= g_first[i].x; v.y *= g_first[i].y; v.z *= g_first[i].z; v.w *= g_first[i].w;
                }
            }
        }
    }

    stage_activations<QT, MT, FUSE>(smem, args, x, M, K, kpad, FUSE ? x_first : nullptr);
    __syncthreads();

    XTile xt;
    xt.qs = reinterpret_cast<const int8_t *>(smem);
    xt.d = reinterpret_cast<const float *>(smem + MT * kpad);
    xt.bs = reinterpret_cast<const int16_t *>(smem + MT * kpad + MT * (kpad / BLK) * 4);
    xt.kt = kpad;
    Dot<QT> xr[MT];
    if (XREG) {
#pragma unroll
        for (int m = 0; m < MT; ++m) xr[m].load_x(xt, m, 0, lane);
    }

    float acc[MT][R];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[m][r] = 0.f;

    // (g, c) = (row group, chunk) cursors; the issue cursor runs one step ahead of the consume
    // cursor and stops on the last step, whose cache lines were just fetched, so every issue is
    // unconditional and no wait ever has to cover a maybe-issued load.
    if constexpr (XREG && (MT == 1 || (MT == 2 && (QT == kTypeQ4_K || QT == kTypeQ8_0Two) && FUSE && !PAIR))) {  // one chunk per row, one or two activation rows: the step index is the row group
        // No load is issued twice (a repeated load of the last step, cheap as it looks, costs 0.4 us of the
        // gate+up launch at one activation row and 0.8 us at two): the loop runs while two more steps follow,
        // the last one or two steps are peeled, and every block still knows exactly which loads are outstanding.
        // (Two rows of the wider formats, of the gate/up pairing and of rows quantized earlier keep the plain loop
        // below: peeled they run out of registers.)
        int g = 0;
        for (; g + 2 < n_groups; g += 2) {
            issue_rows(buf_b, g + 1, 0);
            __builtin_amdgcn_sched_barrier(0);
            consume<QT, MT, R, XREG, PAIR>(buf_a, acc, xr, xt, g, 0, 1, nb, n_rows, row_begin, N, y, M, lane);
            issue_rows(buf_a, g + 2, 0);
            __builtin_amdgcn_sched_barrier(0);
            consume<QT, MT, R, XREG, PAIR>(buf_b, acc, xr, xt, g + 1, 0, 1, nb, n_rows, row_begin, N, y, M, lane);
        }
        if (g + 1 < n_groups) {
            issue_rows(buf_b, g + 1, 0);
            __builtin_amdgcn_sched_barrier(0);
            consume<QT, MT, R, XREG, PAIR>(buf_a, acc, xr, xt, g, 0, 1, nb, n_rows, row_begin, N, y, M, lane);
            consume<QT, MT, R, XREG, PAIR>(buf_b, acc, xr, xt, g + 1, 0, 1, nb, n_rows, row_begin, N, y, M, lane);
        } else if (g < n_groups) {
            consume<QT, MT, R, XREG, PAIR>(buf_a, acc, xr, xt, g, 0, 1, nb, n_rows, row_begin, N, y, M, lane);
        }
        return;
    }
    if (XREG) {  // one chunk per row: the step index is the row group
        for (int g = 0; g < n_groups; g += 2) {
            issue_rows(buf_b, g + 1 < n_groups ? g + 1 : n_groups - 1, 0);
            __builtin_amdgcn_sched_barrier(0);
            consume<QT, MT, R, XREG, PAIR>(buf_a, acc, xr, xt, g, 0, 1, nb, n_rows, row_begin, N, y, M, lane);
            issue_rows(buf_a, g + 2 < n_groups ? g + 2 : n_groups - 1, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (g + 1 < n_groups) consume<QT, MT, R, XREG, PAIR>(buf_b, acc, xr, xt, g + 1, 0, 1, nb, n_rows, row_begin, N, y, M, lane);
        }
        return;
    }
    int ig = 0, ic = 0, cg = 0, cc = 0, issued = 0;
    auto advance = [&](int &g, int &c) {
        c += 1;
        if (c == nch) {
            c = 0;
            g += 1;
        }
    };
    for (int it = 0; it < n_iter; it += 2) {
        if (issued + 1 < n_iter) { advance(ig, ic); ++issued; }
        issue_rows(buf_b, uniform(ig), uniform(ic));
        __builtin_amdgcn_sched_barrier(0);  // keep the loads ahead of the arithmetic that follows
        consume<QT, MT, R, XREG, PAIR>(buf_a, acc, xr, xt, uniform(cg), uniform(cc), nch, nb, n_rows, row_begin, N, y, M, lane);
        advance(cg, cc);
        if (issued + 1 < n_iter) { advance(ig, ic); ++issued; }
        issue_rows(buf_a, uniform(ig), uniform(ic));
        __builtin_amdgcn_sched_barrier(0);
        if (it + 1 < n_iter) {
            consume<QT, MT, R, XREG, PAIR>(buf_b, acc, xr, xt, uniform(cg), uniform(cc), nch, nb, n_rows, row_begin, N, y, M, lane);
            advance(cg, cc);
        }
    }
}


template <int QT, int MT, int R, bool XREG, bool FUSE, bool PAIR = false>
hipError_t launch_decode(const GemvArgs &args, hipStream_t s) {
    constexpr int CH = Geo<QT>::kChunk;
    constexpr int BLK = Geo<QT>::kBlk;
    const int n_targets = PAIR ? 1 : args.n_targets;   // gate and up are walked together: the waves are dealt over the rows of one of them
    if (PAIR && (args.n_targets != 2 || args.t[0].w.N != args.t[1].w.N || args.t[0].w.K != args.t[1].w.K)) return hipErrorInvalidValue;
    int64_t rows_total = 0;
    for (int i = 0; i < n_targets; ++i) rows_total += args.t[i].w.N;
    if (rows_total == 0) return hipSuccess;
    // one workgroup per CU, fewer when there are not enough rows to give every wave one
    static const int wgs_per_cu = tuning_int("QPROJ_DECODE_WGS_PER_CU", 1);
    int64_t grid = (int64_t)cu_count() * wgs_per_cu;
    const int64_t need = (rows_total + kDecodeWaves - 1) / kDecodeWaves;  // at least one row per wave
    if (grid > need) grid = need;
    const int n_waves = (int)grid * kDecodeWaves;
    DecodeArgs a{};
    for (int i = 0; i < kMaxTargets; ++i) a.first_wave[i] = INT_MAX;
    for (int i = 0; i < args.n_targets; ++i) {
        const WeightView &w = args.t[i].w;
        a.N[i] = w.N;
        a.y[i] = args.t[i].y;
        if (QT == kTypeQ4_K) {
            a.p0[i] = w.q4k;
        } else if (QT == kTypeQ6_K) {
            a.p0[i] = w.q6_ql;
            a.p1[i] = w.q6_qh;
            a.p2[i] = reinterpret_cast<const uint8_t *>(w.q6_sc);
            a.p3[i] = reinterpret_cast<const uint8_t *>(w.q6_d);
        } else {
            a.p0[i] = reinterpret_cast<const uint8_t *>(w.q8_qs);
            a.p1[i] = reinterpret_cast<const uint8_t *>(w.q8_d);
        }
    }
    a.qs = args.a.qs;
    a.d = args.a.d;
    a.bsums = args.a.bsums;
    // waves are dealt to the targets in proportion to their rows; a wave never straddles targets
    int given = 0;
    for (int i = 0; i < n_targets; ++i) {
        const int left_after = n_targets - 1 - i;  // every later target gets at least one wave
        int share = (int)((a.N[i] * n_waves + rows_total - 1) / rows_total);
        if (share < 1) share = 1;
        if (i == n_targets - 1 || given + share > n_waves - left_after) share = n_waves - left_after - given;
        if (share < 1) return hipErrorInvalidValue;
        a.first_wave[i] = given;
        const int rpp = (int)((2 * a.N[i] + share - 1) / share);  // rows per pair of waves
        a.rows_per_pair[i] = rpp;
        if ((int64_t)rpp * (int64_t)args.t[i].w.nb * 256 >= ((int64_t)1 << 31)) return hipErrorInvalidValue;  // 32-bit row offsets
        given += share;
    }
    const int64_t K = args.t[0].w.K;
    const int kpad = (int)((K + CH - 1) / CH * CH);
    const size_t smem = (size_t)MT * kpad + (size_t)MT * (kpad / BLK) * 4 + (!is_q8_0<QT> ? (size_t)MT * (kpad / 16) * 2 : 0);
    if (dry_run()) {
        char rows[96] = "";
        for (int i = 0, o = 0; i < n_targets && o < 80; ++i)
            o += snprintf(rows + o, sizeof rows - o, "%s%lld rows/%d a wave pair", i ? ", " : "", (long long)a.N[i], a.rows_per_pair[i]);
        char parts[40] = "";
        if (is_q8_0<QT>) snprintf(parts, sizeof parts, ", %d parts of 1024 weights a step", CH / 1024);
        plan_note("gemv_decode_kernel<%s%s, %d activation rows, %d weight rows a step, activations in %s, %s%s>: grid %lld x %d, %s, LDS %zu B",
                  plan_type_name(args.t[0].w.type), parts, MT, R, XREG ? "registers" : "LDS", FUSE ? "quantizer in the prologue" : "rows quantized earlier",
                  PAIR ? ", gate/up paired + swiglu" : "", (long long)grid, kDecodeThreads, rows, smem);
        return hipSuccess;
    }
    auto kern = &gemv_decode_kernel<QT, MT, R, XREG, FUSE, PAIR>;
    static LdsLimit limit;
    const hipError_t e = limit.allow(kern, smem);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(kDecodeThreads), smem, s, args.x, args.norm_gamma, (int)K, (int)args.t[0].w.nb, kpad, args.M,
                       args.norm_eps, (int)args.norm, a);
    return hipGetLastError();
}

// Q8_0: parts of 1024 weights a step.  Two for rows of at most 2048 (2048 -> 2 x 8192 13.4 -> 10.1 us, 2048 -> 2048 / 512 / 512
// 5.7 -> 4.9 against four, half of whose requests lie past the row), three where they need a quarter fewer parts than steps of
// four (rows of up to 3, 5, 6 and 9 parts).  Four / three, us at 1, 2, 4 rows: 3072 -> 8192 6.3 / 6.0, 7.0 / 6.3, 8.7 / 8.2;
// 5120 -> 13824 15.5 / 14.6, 16.9 / 15.7, 22.6 / 19.9; 9216 -> 4096 8.5 / 7.8, 10.2 / 9.8, 15.8 / 14.4.  Where only a sixteenth goes they
// lose at one and two rows (14336 -> 4096 11.3 / 11.6, 13.7 / 14.2, 21.4 / 21.0; 15360 -> 5120 17.7 / 18.4, 20.7 / 21.4, 29.1 / 28.8) and the
// longer chain of steps costs accuracy.  Error against 64 bits, three over four parts, 2000 outputs a draw, 512 to 1024 draws: 5
// parts 0.982, 6 0.994, 9 0.976; 13 and 14 1.001, 15 1.004, 17 (K = 16896) 1.009, 25 to 29 1.01 to 1.02.
int q8_0_parts(int64_t K) {
    const int64_t n = (K + 1023) / 1024, three = (n + 2) / 3 * 3, four = (n + 3) / 4 * 4;
    return n <= 2 ? 2 : 4 * three <= 3 * four ? 3 : 4;
}

// Rows of one chunk keep their activations in registers, longer ones read the LDS image.  Built are the instances that the
// rule below reaches: two parts are taken for rows that they cover only, steps of two rows in the wider formats likewise.
template <int QT, int MT, int R, bool FUSE, bool PAIR = false>
hipError_t launch_decode_rows(const GemvArgs &args, hipStream_t s) {
    // the wide Q8_0 geometry keeps its 20 activation registers a row only for one row and plain projections (two
    // rows, or the gate/up pairing, would spill), four rows fit in the smallest geometries
    constexpr bool kRegisters = QT == kTypeQ8_0Wide ? MT == 1 && !PAIR : MT <= 2 || QT == kTypeQ4_K || QT == kTypeQ8_0Two;
    if constexpr (kRegisters)
        if (args.t[0].w.K <= Geo<QT>::kChunk) return launch_decode<QT, MT, R, true, FUSE, PAIR>(args, s);
    if constexpr (QT != kTypeQ8_0Two && (QT == kTypeQ4_K || R == 1 || PAIR)) return launch_decode<QT, MT, R, false, FUSE, PAIR>(args, s);
    return hipErrorInvalidValue;   // (a chunk too long for an instance that is never asked for it)
}

template <int QT, bool FUSE>
hipError_t launch_decode_mt(const GemvArgs &args, int mt, hipStream_t s) {
    if (args.swiglu_pair) {
        if (mt == 1) return launch_decode_rows<QT, 1, 2, FUSE, true>(args, s);
        if (mt == 2) return launch_decode_rows<QT, 2, 2, FUSE, true>(args, s);
        return hipErrorInvalidValue;
    }
    // two rows per step only when every wave has at least two rows to walk (with 1.5 rows per wave, split
    // 2 + 1 over a pair of waves, two-row steps measured slower: q/k/v 7.4 against 6.4 us; with one row a wave
    // a two-row step fetches that row twice)
    int64_t rows_total = 0;
    for (int i = 0; i < args.n_targets; ++i) rows_total += args.t[i].w.N;
    static const int two_rows_env = tuning_int("QPROJ_DECODE_TWO_ROWS", -1);
    const bool pairs = two_rows_env >= 0 ? two_rows_env != 0 : rows_total >= (int64_t)2 * cu_count() * kDecodeWaves;
    // Two activation rows, or rows of several chunks, in the wider formats walk one weight row a step whatever the row count:
    // their two-row steps run out of registers (two rows, Q6_K 4096 -> 14336 17.5 -> 13.9 us, Q8_0 8192 x 8192 20.1 -> 17.6; one
    // row, 8192 x 8192 Q8_0 19.2 -> 16.9, Q6_K 15.6 -> 14.3).  The two-part Q8_0 steps are as small as Q4_K's.
    constexpr bool kSmall = QT == kTypeQ4_K || QT == kTypeQ8_0Two;
    switch (mt) {
    case 1:
        if constexpr (!kSmall)
            if (args.t[0].w.K > Geo<QT>::kChunk) return launch_decode_rows<QT, 1, 1, FUSE>(args, s);
        return pairs ? launch_decode_rows<QT, 1, 2, FUSE>(args, s) : launch_decode_rows<QT, 1, 1, FUSE>(args, s);
    case 2:
        if constexpr (kSmall)
            if (pairs) return launch_decode_rows<QT, 2, 2, FUSE>(args, s);
        return launch_decode_rows<QT, 2, 1, FUSE>(args, s);
    case 4: return launch_decode_rows<QT, 4, 1, FUSE>(args, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

int cu_count() {
    if (plan_cu_count() > 0) return plan_cu_count();
    static int n = [] {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
        return v;
    }();
    return n;
}

bool decode_kernel_norm_fits(int mt, int64_t K) {
    return mt >= 1 && mt <= 4 && K <= (int64_t)256 * kDecodeWaves * prefetched_pieces(mt);
}

// the largest K whose activation rows fit the LDS image (mt rows)
bool decode_kernel_fits(int type, int mt, int64_t K) {
    const int ch = 4096;
    const int blk = type == kTypeQ8_0 ? 32 : 256;
    const int64_t kpad = (K + ch - 1) / ch * ch;
    const int64_t smem = mt * kpad + mt * (kpad / blk) * 4 + (type != kTypeQ8_0 ? mt * (kpad / 16) * 2 : 0);
    return mt <= 4 && smem <= 96 * 1024;
}

hipError_t launch_gemv_decode(const GemvArgs &args, int mt, bool fuse_quantize, hipStream_t s) {
    switch (args.t[0].w.type) {
    case kTypeQ4_K: return fuse_quantize ? launch_decode_mt<kTypeQ4_K, true>(args, mt, s) : launch_decode_mt<kTypeQ4_K, false>(args, mt, s);
    case kTypeQ6_K: return fuse_quantize ? launch_decode_mt<kTypeQ6_K, true>(args, mt, s) : launch_decode_mt<kTypeQ6_K, false>(args, mt, s);
    case kTypeQ8_0:
        switch (q8_0_parts(args.t[0].w.K)) {
        case 2: return fuse_quantize ? launch_decode_mt<kTypeQ8_0Two, true>(args, mt, s) : launch_decode_mt<kTypeQ8_0Two, false>(args, mt, s);
        case 3: return fuse_quantize ? launch_decode_mt<kTypeQ8_0Three, true>(args, mt, s) : launch_decode_mt<kTypeQ8_0Three, false>(args, mt, s);
        default: break;
        }
        return fuse_quantize ? launch_decode_mt<kTypeQ8_0Wide, true>(args, mt, s) : launch_decode_mt<kTypeQ8_0Wide, false>(args, mt, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace qproj
