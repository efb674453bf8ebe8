// Prefill projection: Q4_K weights x per-32 int8 activations on the int8 matrix cores.
//
//   y[m][n] = sum_blk (d_n*sc_{n,blk}) * da_{m,blk} * I_{m,n,blk}  -  sum_blk (dmin_n*mn_{n,blk}) * (da_{m,blk}*isum_{m,blk})
//   I_{m,n,blk} = sum over the 32 weights of the sub-block of q * a      (exact, int32)
//
// A workgroup owns a 128 (tokens) x 128 (weight rows) tile; each of its 8 waves a 32x64
// sub-tile = two v_mfma_i32_32x32x32_i8 products per 32-wide sub-block.  Both operands change
// scale every 32 K-elements, so an int32 accumulator is meaningful for ONE product only: each
// product is folded into the fp32 accumulators right away.  That fp32 work, not the matrix cores,
// bounds this kernel (the vector ALU issues in 94 % of its cycles; at this load the clock sinks to
// 1.8 GHz), so everything else is kept off the vector ALU:
//   - two instructions an output and block instead of three (see `product`);
//   - activations go from global memory straight into LDS, addresses are one register an operand
//     and immediate offsets, the four sub-blocks of a K-step are unrolled;
//   - the min term is a separate small GEMM over K/32 (activation block sums x mins) done on the
//     fp16 matrix cores before the main loop, with both operands split into fp16 high and low
//     parts (the mins are 17-bit products, split exactly; the sums keep 22 bits);
//   - LDS holds only the two int8 operand tiles and the transposed scales, double buffered over
//     K-steps of 128 so that the global loads of step s+1 overlap step s.
// Measured, three instructions and operands through registers -> this, same card in turn:
// 4096 x 4096 against 14336 rows 783 -> 684 us (614 -> 703 TOPS), 61.5 -> 41.2 vector instructions beside a product.
#include <cstdlib>
#include <type_traits>
#include "gemm_convert.h"
#include "qproj_device.h"
#include "qproj_internal.h"
#include "gemm_tiles.h"
#include "lds_direct.h"

namespace qproj {

namespace {

constexpr int BM = 128, BN = 128, BK = 128;

// Rows of 128 bytes; the 16-byte segment `seg` of row r sits in slot seg ^ ((r / 2) % 8) (a load straight into LDS
// cannot pad rows; 16 consecutive rows reading the same segment hit 16 different quadwords of the 64 banks).
struct GemmStage {
    int8_t a[BM * BK];   // activations  [m][k]
    int8_t b[BN * BK];   // weights      [n][k], nibbles expanded
    float sc[8][BM];     // 0..3: da [sub-block][m]; 4..7: d*sc (Q8_0: d) [sub-block][n]
};
static_assert(BM == BN, "one array of scales");

struct GemmSmem {
    GemmStage st[2];
};

// registers one thread carries from global memory to LDS for one K-step
struct StageRegs {
    v4i wq;   // Q4_K: 16 nibble bytes of a weight row
    v4i ad;   // threads 0..127: activation scales; threads 128..255: block header (Q8_0: four scales) of a weight row
};

__device__ __forceinline__ void split_h(float v, _Float16 &hi, _Float16 &lo) {
    hi = (_Float16)v;
    lo = (_Float16)(v - (float)hi);
}

constexpr int kGemmThreads = 512;
constexpr float kMagic = 12582912.f;   // 1.5 * 2^23: one integer step is one step of the float

// QT = Q4_K: per-32 int8 activations with fp32 scales and block sums (the prefill format).
// QT = Q8_0: ggml's Q8_0 activation blocks against Q8_0 weights: the same product without nibbles,
// without a min term, and with a weight scale per 32 instead of d*sc per sub-block.
// K of a matrix goes in n_split equal stretches (whole super-blocks for Q4_K); with more than one the tiles go to
// out[stretch][M][N] and an adding pass puts the stretches together in order.  The matrices of a call (q/k/v, gate/up)
// share a launch: at 33 .. 256 tokens one of them alone leaves most of the chip's 512 places (two workgroups a compute
// unit) empty, and every launch pays the latency of its K loop again.  Four layers of 3072 / 1024 / 8192 Q8_0 weights
// at 187 tokens, a launch and an adding pass a matrix -> this: 828 -> 564 .. 579 us.
struct Per32Target {
    WeightView w;
    float *out;   // the output, or [n_split][M][N] partial tiles
    int tiles_pad, n_split, first_wg;   // tiles_pad: workgroups of one stretch, a multiple of the 8 XCDs
};
struct Per32Args {
    int n;
    Per32Target t[kMaxTargets];
    ActView a;
    int64_t M;
};
template <int QT>
__global__ __launch_bounds__(kGemmThreads, 4) void gemm_per32_kernel(const Per32Args g) {
    constexpr bool kQ4 = QT == kTypeQ4_K;
    extern __shared__ __align__(16) uint8_t smem_raw[];
    GemmSmem &sm = *reinterpret_cast<GemmSmem *>(smem_raw);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;  // 4 x 2 waves
    int ti = 0;
    if constexpr (!kQ4) {   // (Q4_K launches carry one matrix)
#pragma unroll
        for (int i = 1; i < kMaxTargets; ++i)
            if (i < g.n && (int)blockIdx.x >= g.t[i].first_wg) ti = i;
    }
    const Per32Target &t = g.t[ti];
    const WeightView w = t.w;
    const ActView a = g.a;
    const int64_t N = w.N, K = w.K, M = g.M;
    const int tiles_n = (int)((N + BN - 1) / BN), tiles_m = (int)((M + BM - 1) / BM);
    int split = 0, pid = (int)blockIdx.x - t.first_wg;
    if (t.n_split > 1) {
        split = pid / t.tiles_pad;
        pid -= split * t.tiles_pad;
    }
    if (pid >= tiles_n * tiles_m) return;   // padding: the whole workgroup leaves
    int tile_n, tile_m;
    tile_of_workgroup(tiles_n, tiles_m, pid, tile_n, tile_m);
    const int64_t n0 = (int64_t)tile_n * BN, m0 = (int64_t)tile_m * BM;
    const int64_t kb32 = K / 32;
    const int l32 = lane & 31, lh = lane >> 5;
    // this workgroup's stretch of K, in units of 256 (Q4_K super-blocks; two K-steps)
    const int64_t n_units = (K + 255) / 256, per = (n_units + t.n_split - 1) / t.n_split;
    const int64_t u_begin = min((int64_t)split * per, n_units), u_end = min(u_begin + per, n_units);
    float *const y = t.out + (size_t)split * M * N;

    v16f acc[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[j][v] = 0.f;

    // ---------------------------------------------------------------- min term on the fp16 cores
    // acc = -(1/prescale) * sum_kb A[m][kb] * B[n][kb] is built as +sum with negated B and scaled later.
    // The activation side (d * block sum, as fp16 high and low parts) comes ready from the quantizer.  The
    // weight side (-dmin * min of every sub-block, split the same way) is worked out once per workgroup,
    // 16 super-blocks at a time, into the LDS the main loop will use afterwards: two planes
    // [super-block][row][8 x fp16], so that every wave only reads operands and issues matrix instructions.
    if constexpr (kQ4) {
        constexpr int SBC = 16;                                   // super-blocks per pass (2 x 16 x 128 x 16 B = 64 KB)
        static_assert(2 * SBC * BN * 16 <= (int)sizeof(GemmSmem), "the min-term planes must fit the main loop's LDS");
        uint8_t *plane_hi = smem_raw, *plane_lo = smem_raw + SBC * BN * 16;
        const int64_t mrow = m0 + wm * 32 + l32 < M ? m0 + wm * 32 + l32 : M - 1;   // rows past M are never stored
        for (int64_t c0 = u_begin; c0 < u_end; c0 += SBC) {
            const int nsbc = (int)(u_end - c0 < SBC ? u_end - c0 : SBC);
            if (c0 > u_begin) __syncthreads();   // the previous pass has been read
            for (int base = 0; base < BN * nsbc; base += 4 * kGemmThreads) {
                v4i hd[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {   // four headers in flight per thread
                    const int item = min(base + u * kGemmThreads + tid, BN * nsbc - 1);
                    int64_t n = n0 + (item & (BN - 1));
                    if (n >= N) n = N - 1;
                    hd[u] = *reinterpret_cast<const v4i *>(w.q4k + (n * w.nb + c0 + (item >> 7)) * 144);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int item = base + u * kGemmThreads + tid;
                    if (item >= BN * nsbc) continue;
                    const ScalesK4 sc = unpack_scales_k4((uint32_t)hd[u][1], (uint32_t)hd[u][2], (uint32_t)hd[u][3]);
                    const float dmin = h2f((uint32_t)hd[u][0] >> 16);
                    v8h bh, bl;
#pragma unroll
                    for (int t = 0; t < 8; ++t) {
                        _Float16 h, l;
                        split_h(-(dmin * (float)min_k4(sc, t)), h, l);
                        bh[t] = h;
                        bl[t] = l;
                    }
                    *reinterpret_cast<v8h *>(plane_hi + item * 16) = bh;   // item = super-block * 128 + row
                    *reinterpret_cast<v8h *>(plane_lo + item * 16) = bl;
                }
            }
            __syncthreads();
            const int n_steps = (nsbc + 1) / 2;   // 16 sub-blocks = two super-blocks per product
            v8h ah, al, ah_n, al_n;
            auto load_a = [&](v8h &h, v8h &l, int s) {
                int sbl = 2 * s + lh;
                if (sbl >= nsbc) sbl = nsbc - 1;   // past the end: any finite operand, the weight side is zero there
                const v8h *mp = reinterpret_cast<const v8h *>(a.msum + (mrow * w.nb + c0 + sbl) * 16);
                h = mp[0];
                l = mp[1];
            };
            load_a(ah, al, 0);
            for (int s = 0; s < n_steps; ++s) {
                load_a(ah_n, al_n, s + 1 < n_steps ? s + 1 : s);   // in flight during this step
                const int sbl = 2 * s + lh;
                const bool live = sbl < nsbc;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int o = ((live ? sbl : 0) * BN + wn * 64 + j * 32 + l32) * 16;
                    v8h bh = *reinterpret_cast<const v8h *>(plane_hi + o);
                    v8h bl = *reinterpret_cast<const v8h *>(plane_lo + o);
                    if (!live) {
#pragma unroll
                        for (int t = 0; t < 8; ++t) bh[t] = bl[t] = (_Float16)0.f;
                    }
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh, acc[j], 0, 0, 0);
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl, acc[j], 0, 0, 0);
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh, acc[j], 0, 0, 0);
                }
                ah = ah_n;
                al = al_n;
            }
        }
        // the operand was normalised by the row (rs[m], a power of two) and pre-scaled by 1/16: both undone exactly
        __syncthreads();   // the planes have been read
        float *rs_tile = reinterpret_cast<float *>(smem_raw);   // the tile's 128 row normalisers, times 16
        if (tid < BM) rs_tile[tid] = a.rs[m0 + tid < M ? m0 + tid : M - 1] * (1.0f / kMinPrescale);
        __syncthreads();
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const float4 f = *reinterpret_cast<const float4 *>(rs_tile + wm * 32 + 8 * g + 4 * lh);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                acc[j][4 * g] *= f.x; acc[j][4 * g + 1] *= f.y; acc[j][4 * g + 2] *= f.z; acc[j][4 * g + 3] *= f.w;
            }
        }
        __syncthreads();   // the main loop may overwrite the tile
    }

    // ---------------------------------------------------------------- main loop, int8 cores
    // Addresses: a scalar base per operand plus a 32-bit lane offset that never changes; the K position is added
    // to the scalar side.  (64-bit pointers per lane cost the registers this kernel does not have.)  Rows past the
    // end of a tile read the last valid row: their results are never stored.
    const int mrow_cap = (int)(M - 1 - m0 < BM - 1 ? M - 1 - m0 : BM - 1);
    const int nrow_cap = (int)(N - 1 - n0 < BN - 1 ? N - 1 - n0 : BN - 1);
    const int8_t *abase_s = scalar_pointer(a.qs + m0 * K);
    const global_ptr<float> adbase_s = scalar_global(a.d + m0 * kb32);
    // requests straight into LDS: chunk wave + 8*i of a tile = its rows 8*(wave + 8*i) .. +7
    const int swave = __builtin_amdgcn_readfirstlane(wave);
    const int seg = (lane & 7) ^ ((lane >> 4) | ((swave & 1) << 2));   // slot lane%8 of row r holds segment slot ^ (r/2)%8
    uint32_t aoffg[2], w8offg[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = 8 * (wave + 8 * i) + (lane >> 3);
        aoffg[i] = (uint32_t)(row < mrow_cap ? row : mrow_cap) * (uint32_t)K + 16u * seg;
        w8offg[i] = (uint32_t)(row < nrow_cap ? row : nrow_cap) * (uint32_t)K + 16u * seg;   // Q8_0 only
    }
    // threads 0..127: byte offset of a token's activation scales; 128..255: of a weight row's header (Q8_0: scales)
    global_ptr<uint8_t> wbase_s = nullptr;
    const int8_t *w8base_s = nullptr;
    global_ptr<uint16_t> w8d_s = nullptr;
    uint32_t woffg = 0, doffg = (uint32_t)min(tid, mrow_cap) * (uint32_t)kb32 * 4u;
    if constexpr (kQ4) {
        wbase_s = scalar_global(w.q4k + n0 * w.nb * 144);
        woffg = (uint32_t)min(tid >> 2, nrow_cap) * (uint32_t)w.nb * 144u + 16u + 16u * (tid & 3);
        if (tid >= BM) doffg = (uint32_t)min(tid - BM, nrow_cap) * (uint32_t)w.nb * 144u;
    } else {
        w8base_s = scalar_pointer(w.q8_qs + n0 * K);
        w8d_s = scalar_global(w.q8_d + n0 * w.nb);
        if (tid >= BM) doffg = (uint32_t)min(tid - BM, nrow_cap) * (uint32_t)w.nb * 2u;
    }
    // the half of a super-block a K-step is (its parity) is known at compile time
    auto load_stage = [&](StageRegs &r, uint32_t ks, auto parity) {
        constexpr int P = decltype(parity)::value;
        GemmStage &st = sm.st[P];
#pragma unroll
        for (int i = 0; i < 2; ++i)   // activations: 128 rows x 128 B
            global_to_lds16(abase_s + (aoffg[i] + ks * BK), st.a + (swave + 8 * i) * 1024);
        if constexpr (kQ4) {  // weights: 128 rows x 64 packed bytes (two 64-weight chunks of the super-block)
            r.wq = load_global<v4i>(wbase_s, woffg + ((ks >> 1) * 144u + 64u * P));
        } else {              // weights: 128 rows x 128 int8
#pragma unroll
            for (int i = 0; i < 2; ++i) global_to_lds16(w8base_s + (w8offg[i] + ks * BK), st.b + (swave + 8 * i) * 1024);
        }
        if (swave < 4) {   // scalar branches: one base, one lane offset
            if (kQ4 || swave < 2) {
                r.ad = load_global<v4i>(swave < 2 ? (global_ptr<uint8_t>)adbase_s : wbase_s, doffg + (swave < 2 ? ks * 16u : (ks >> 1) * 144u));
            } else {           // the four fp16 scales of this K-step
                const v2i d4 = load_global<v2i>(w8d_s, doffg + ks * 8u);
                r.ad[0] = d4[0];
                r.ad[1] = d4[1];
            }
        }
    };
    auto store_stage = [&](const StageRegs &r, auto parity) {
        constexpr int P = decltype(parity)::value;
        GemmStage &st = sm.st[P];
        if constexpr (kQ4) {
            // 16 packed bytes = bytes 16*(part&1).. of chunk (part>>1): low nibbles -> sub-block 2c, high -> 2c+1
            const int row = tid >> 2, part = tid & 3, slot = ((part >> 1) * 4 + (part & 1)) ^ ((row >> 1) & 7);
            int8_t *base = st.b + row * BK;
            v4i lo, hi;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                lo[c] = r.wq[c] & 0x0f0f0f0f;
                hi[c] = (int)((uint32_t)r.wq[c] >> 4) & 0x0f0f0f0f;
            }
            *reinterpret_cast<v4i *>(base + 16 * slot) = lo;
            *reinterpret_cast<v4i *>(base + 16 * (slot ^ 2)) = hi;
        }
        float *const dst = &st.sc[0][0] + tid;   // (thread BM + i: entry i of rows 1.. , so rows 4..7 are three further on)
        if (swave < 2) {
#pragma unroll
            for (int t = 0; t < 4; ++t) dst[t * BM] = __int_as_float(r.ad[t]);
        } else if (swave < 4) {
            if constexpr (kQ4) {
                const ScalesK4 sc = unpack_scales_k4((uint32_t)r.ad[1], (uint32_t)r.ad[2], (uint32_t)r.ad[3]);
                const float d = h2f((uint32_t)r.ad[0]);
#pragma unroll
                for (int t = 0; t < 4; ++t) dst[(3 + t) * BM] = d * (float)scale_k4(sc, 4 * P + t);
            } else {
#pragma unroll
                for (int t = 0; t < 4; ++t) dst[(3 + t) * BM] = h2f(((uint32_t)r.ad[t >> 1] >> (16 * (t & 1))) & 0xffffu);
            }
        }
    };

    // Q4_K: the integer sums leave the matrix instruction as the bits of the float kMagic + I (its addend is kMagic's
    // bits), and (kMagic + I) * w - kMagic * w in one fma is I * w rounded once: kMagic * w is exact, w = fp16 scale x
    // 6-bit sub-block scale has 17 significant bits, |I| < 2^16.  Two vector instructions an output and block where
    // int -> float, scale product and fma are three, and as many roundings.  For Q8_0 they are one rounding more, since
    // the product of its two fp16 scales is exact: it keeps the three.
    v16i addend;
#pragma unroll
    for (int v = 0; v < 16; ++v) addend[v] = kQ4 ? __float_as_int(kMagic) : 0;
    if constexpr (kQ4) asm volatile("" : "+v"(addend));   // in registers: rebuilt for every product it costs eight moves
    auto product = [&](const v4i &af, const v4i &bf, float ws, const v4i (&ad)[4], float (&sum)[16]) {
        const v16i I = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, bf, addend, 0, 0, 0);
        const float nws = -kMagic * ws;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const float da = __int_as_float(ad[v >> 2][v & 3]);
            sum[v] = kQ4 ? fmaf(fmaf(__int_as_float(I[v]), ws, nws), da, sum[v]) : fmaf((float)I[v], da * ws, sum[v]);
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) asm volatile("" : "+v"(sum[v]));
    };
    const uint32_t ks_begin = (uint32_t)u_begin * 2, ks_end = (uint32_t)min(u_end * 2, K / BK);
    float sum[2][16];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) sum[j][v] = acc[j][v];
    // segment 2*kb + lh of row l%32 (of the wave's tokens, of its first 32 weight rows): offset ^ 32*kb
    int fa = (wm * 32 + l32) * BK + 16 * (lh ^ ((l32 >> 1) & 7)), fb = (wn * 64 + l32) * BK + 16 * (lh ^ ((l32 >> 1) & 7));
    StageRegs regs;
    auto step = [&](uint32_t ks, auto parity) {
        constexpr int P = decltype(parity)::value;
        const std::integral_constant<int, 1 - P> other{};
        const GemmStage &st = sm.st[P];
        const bool more = ks + 1 < ks_end;
        if (more) load_stage(regs, ks + 1, other);   // in flight during the arithmetic below
        asm volatile("" : "+v"(fa), "+v"(fb));   // the eight addresses are worked out on the spot, not kept in registers
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            const v4i af = *reinterpret_cast<const v4i *>(st.a + (fa ^ (32 * kb)));
            const v4i bf0 = *reinterpret_cast<const v4i *>(st.b + (fb ^ (32 * kb)));
            const v4i bf1 = *reinterpret_cast<const v4i *>(st.b + (fb ^ (32 * kb)) + 32 * BK);
            const float w0 = st.sc[4 + kb][wn * 64 + l32], w1 = st.sc[4 + kb][wn * 64 + 32 + l32];
            v4i ad[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) ad[g] = *reinterpret_cast<const v4i *>(&st.sc[kb][wm * 32 + 8 * g + 4 * lh]);
            // (the empty asm statements keep the sums of a block together: left alone the compiler postpones the last
            // fma of every output and spills hundreds of registers)
            product(af, bf0, w0, ad, sum[0]);
            product(af, bf1, w1, ad, sum[1]);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (more) store_stage(regs, other);
        __syncthreads();   // (waits for the requests into LDS as well)
    };
    if (ks_begin < ks_end) {
        load_stage(regs, ks_begin, std::integral_constant<int, 0>{});
        store_stage(regs, std::integral_constant<int, 0>{});
    }
    __syncthreads();
    for (uint32_t ks = ks_begin; ks < ks_end; ks += 2) {
        step(ks, std::integral_constant<int, 0>{});
        if (ks + 1 < ks_end) step(ks + 1, std::integral_constant<int, 1>{});
    }

    // ---- store: accumulator register v of lane l is row 8*(v/4) + 4*(l/32) + v%4, column l%32
    // (the lane's coordinates are worked out again from the thread index, made opaque so that nothing of the
    // address arithmetic is carried through the main loop in registers the loop needs)
    int tid_s = tid;
    asm volatile("" : "+v"(tid_s));
    const int l32_s = tid_s & 31, lh_s = (tid_s >> 5) & 1, wm_s = tid_s >> 7, wn_s = (tid_s >> 6) & 1;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int64_t n = n0 + wn_s * 64 + j * 32 + l32_s;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int64_t m = m0 + wm_s * 32 + 8 * (v >> 2) + 4 * lh_s + (v & 3);
            if (m < M && n < N) y[m * N + n] = sum[j][v];
        }
    }
}

// ------------------------------------------------------------------------------------------------
// ggml activation format (Q8_K: one scale per 256) x Q4_K on the int8 matrix cores.
//
// With a single activation scale per super-block the integer sums of its eight sub-blocks may be
// added before anything turns into floating point; only the 6-bit sub-block scale sc stands in the
// way, and sc*q (up to 945) does not fit an int8 operand.  Written in base 8, sc = 8*sc_hi + sc_lo,
// both products sc_lo*q and sc_hi*q stay below 106: two int8 weight operands and two accumulation
// chains over the whole super-block run entirely inside the matrix cores,
//     I_lo = sum_k (sc_lo*q) * a,   I_hi = sum_k (sc_hi*q) * a,   sum_k sc*q*a = 8*I_hi + I_lo,
// so the vector ALU only works once per 256 weights (shift-add, int->float, one fma with dx*d).
// Twice the matrix instructions of the per-32 kernel, a third of its vector instructions.
// The weights never become an LDS tile: they are converted in registers.  Inside a super-block
// the order of the 256 products is free (both chains run over all of it), so a lane may feed the matrix
// instruction with whichever 16 weights it likes as long as the activation operand carries the
// matching 16: lane (row l%32, half l/32) takes the 64 contiguous nibble bytes [64*half, 64*half+64)
// of its own weight row = sub-blocks 4*half .. 4*half+3, expands and scales them in registers, and
// reads the activations of exactly those sub-blocks from LDS.  Each of the NW waves owns 32 weight
// rows of the tile and all of its 64 tokens.
//
// Memory side: a lane-per-row load touches 64 cache lines per instruction and the vector memory
// pipeline, not the arithmetic, becomes the limit.  So every wave fetches its 32 raw 144-byte blocks
// with consecutive lanes on consecutive 16-byte pieces (288 pieces, five loads), parks them in a
// wave-private LDS strip exactly as they lie in memory (a row stride of 144 bytes is conflict-free
// for 16-byte reads) and picks its row's header and nibbles out of the strip.  The min term rides
// along: the activation quantizer has already written d*(sub-block sum)/16 as fp16 pairs, the tile
// of those is staged with the activations, and two fp16 matrix instructions per super-block and
// token tile (operand [high | low] against [-dmin*min high | same], then [high | low] against
// [-dmin*min low | 0]) add it to the accumulators, which therefore run in units of 1/16 until the
// final store.  One workgroup barrier per 256 weights.
constexpr int DLA = 256 + 16;   // LDS row stride of the activation tile in bytes

template <int NW>
struct DirectSmem {
    int8_t a[2][64 * DLA];           // activations of one super-block [token][256 + pad]
    uint16_t ms[2][64 * 16];         // min-term operand [token][8 high | 8 low] (fp16 bits)
    float dx[2][64];                 // activation scale of the super-block
    uint8_t park[NW][32 * 144];      // per wave: the raw blocks of its 32 weight rows
};

struct DirectB {     // one super-block of the lane's weight row
    v4i hdr;         // d, dmin, 12 bytes of 6-bit scales and mins
    v4i q[4];        // 64 nibble bytes: q[2*gg + half] = bytes 16*half.. of the 32-byte group 2*(l/32) + gg
};

// Up to three matrices that multiply the same activation rows (q/k/v, gate/up) ride in one launch: a matrix of
// 1024 rows against 512 tokens is 64 tiles, an eighth of the workgroups the chip holds, and took as long alone
// as the 4096-row one beside it.  Each matrix owns a run of workgroups that starts at a multiple of 8.
struct DirectTargets {
    int n;
    WeightView w[3];
    float *y[3];
    int first_wg[3];
};

template <int NW>
__global__ __launch_bounds__(64 * NW, 2) void gemm_q4k_q8k_direct_kernel(const DirectTargets tg, const ActView a, int64_t M,
                                                                        float *__restrict__ part) {
    constexpr int NT = 64 * NW, TN = 32 * NW;
    constexpr int PA = 1024 / NT;   // 16-byte activation pieces a thread moves per super-block
    extern __shared__ __align__(16) uint8_t smem_raw[];
    DirectSmem<NW> &sm = *reinterpret_cast<DirectSmem<NW> *>(smem_raw);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    WeightView w = tg.w[0];
    float *__restrict__ y = tg.y[0];
    int first_wg = 0;
#pragma unroll
    for (int i = 1; i < 3; ++i)
        if (i < tg.n && (int)blockIdx.x >= tg.first_wg[i]) {
            w = tg.w[i];
            y = tg.y[i];
            first_wg = tg.first_wg[i];
        }
    const int64_t N = w.N, K = w.K, nb = w.nb;
    int tile_n, tile_m;
    {
        const int tiles_n = (int)((N + TN - 1) / TN), tiles_m = (int)((M + 63) / 64), pid = (int)blockIdx.x - first_wg;
        if (pid >= tiles_n * tiles_m) return;   // padding between two matrices: the whole workgroup leaves
        tile_of_workgroup(tiles_n, tiles_m, pid, tile_n, tile_m);
    }
    const int64_t n0 = (int64_t)tile_n * TN, m0 = (int64_t)tile_m * 64;
    const int l32 = lane & 31, lh = lane >> 5;

    v16f acc[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[j][v] = 0.f;

    // ---- global -> register -> LDS plumbing.  Every address is a wave-uniform base plus a 32-bit
    // lane offset; rows past the edge of the matrix repeat the last valid row (never stored).
    // weights: piece p = lane + 64*c of the wave's 288 -> row p / 9, 16-byte part p % 9
    const int64_t wave_row0 = n0 + wave * 32 < N ? n0 + wave * 32 : N - 1;
    const int wrow_cap = (int)(N - 1 - wave_row0 < 31 ? N - 1 - wave_row0 : 31);
    const uint8_t *wbase = w.q4k + wave_row0 * nb * 144;
    uint32_t woff[5];
    int wpark[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) {
        const int p = lane + 64 * c < 287 ? lane + 64 * c : 287;
        const int r = p / 9 < wrow_cap ? p / 9 : wrow_cap;
        woff[c] = (uint32_t)(r * (int)nb * 144 + 16 * (p % 9));
        wpark[c] = 16 * p;
    }
    // activations: piece id = tid + NT*p -> token id / 16, 16-byte segment id % 16
    const int mrow_cap = (int)(M - 1 - m0 < 63 ? M - 1 - m0 : 63);
    const int8_t *abase = a.qs + m0 * K;
    uint32_t aoffg[PA];
    int aoffl[PA];
#pragma unroll
    for (int p = 0; p < PA; ++p) {
        const int id = tid + NT * p, row = id >> 4, seg = id & 15;
        aoffg[p] = (uint32_t)((row < mrow_cap ? row : mrow_cap) * (int)K + 16 * seg);
        aoffl[p] = row * DLA + 16 * seg;
    }
    // min-term operand: 64 tokens x 32 bytes, thread t (mod 128) moves 16 bytes; scale: thread t (mod 64)
    const uint8_t *msbase = reinterpret_cast<const uint8_t *>(a.msum) + m0 * nb * 32;
    const int msrow = (tid & 127) >> 1;
    const uint32_t msoffg = (uint32_t)((msrow < mrow_cap ? msrow : mrow_cap) * (int)nb * 32 + 16 * (tid & 1));
    const float *dxbase = a.d + m0 * nb;
    const uint32_t dxoffg = (uint32_t)(((tid & 63) < mrow_cap ? (tid & 63) : mrow_cap) * (int)nb);
    // the min-term operand is normalised by the row (rs[m], a power of two): the accumulators run in units of
    // 1 / (16 * rs[m]) until the store, so the activation scales are divided by rs[m] as they are staged (exact)
    const float rs_mine = a.rs[m0 + ((tid & 63) < mrow_cap ? (tid & 63) : mrow_cap)];
    const float inv_rs = 1.0f / rs_mine;

    v4i stg[5], areg[PA], msreg;
    float dxreg;
    auto load_next = [&](int64_t sb) {   // activations first: they are wanted at the end of this trip already
#pragma unroll
        for (int p = 0; p < PA; ++p) areg[p] = *reinterpret_cast<const v4i *>(abase + sb * 256 + aoffg[p]);
        msreg = *reinterpret_cast<const v4i *>(msbase + sb * 32 + msoffg);
        dxreg = dxbase[sb + dxoffg];
#pragma unroll
        for (int c = 0; c < 5; ++c) stg[c] = *reinterpret_cast<const v4i *>(wbase + sb * 144 + woff[c]);
    };
    uint8_t *park = sm.park[wave];
    auto store_next = [&](int buf) {
#pragma unroll
        for (int p = 0; p < PA; ++p) *reinterpret_cast<v4i *>(sm.a[buf] + aoffl[p]) = areg[p];
        // threads beyond the first 128 / 64 repeat a store of the same value: no branch, no load sunk into one
        *reinterpret_cast<v4i *>(reinterpret_cast<uint8_t *>(sm.ms[buf]) + 16 * (tid & 127)) = msreg;
        sm.dx[buf][tid & 63] = dxreg * inv_rs;   // (here, not at the load: nothing waits for the load before it must)
#pragma unroll
        for (int c = 0; c < 5; ++c) *reinterpret_cast<v4i *>(park + wpark[c]) = stg[c];
    };

    const v16i zi = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    auto superblock = [&](const DirectB &b, int buf) {
        const ScalesK4 sc = unpack_scales_k4((uint32_t)b.hdr[1], (uint32_t)b.hdr[2], (uint32_t)b.hdr[3]);
        // ---- min term: -dmin*min of the 8 sub-blocks as fp16 high and low parts
        {
            const float ndmin = -h2f((uint32_t)b.hdr[0] >> 16);
            v8h bh, bl;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                _Float16 h, l;
                split_h(ndmin * (float)min_k4(sc, t), h, l);
                bh[t] = h;
                bl[t] = lh ? (_Float16)0.f : l;
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const v8h am = *reinterpret_cast<const v8h *>(reinterpret_cast<const uint8_t *>(sm.ms[buf]) +
                                                             (j * 32 + l32) * 32 + 16 * lh);
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(am, bh, acc[j], 0, 0, 0);
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(am, bl, acc[j], 0, 0, 0);
            }
        }
        // ---- the lane's four sub-block scales, split in base 8 and spread over both 16-bit halves
        const uint32_t scw = lh ? sc.sc_hi : sc.sc_lo;
        const uint32_t lo_w = scw & 0x07070707u, hi_w = (scw >> 3) & 0x07070707u;
        const int8_t *ap = sm.a[buf] + l32 * DLA + 128 * lh;
        v16i ilo[2], ihi[2];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int gg = t >> 2, nib = (t >> 1) & 1, half = t & 1, i = 2 * gg + nib;
            const uint32_t sl = byte_to_u16x2(lo_w, i), sh = byte_to_u16x2(hi_w, i);
            const v4i raw = b.q[2 * gg + half];
            v4i bl, bh;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint32_t x = nib ? ((uint32_t)raw[c] >> 4) & 0x0f0f0f0fu : (uint32_t)raw[c] & 0x0f0f0f0fu;
                bl[c] = (int)pk_mul_u16(x, sl);
                bh[c] = (int)pk_mul_u16(x, sh);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const v4i af = *reinterpret_cast<const v4i *>(ap + j * 32 * DLA + 32 * i + 16 * half);
                ilo[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, bl, t == 0 ? zi : ilo[j], 0, 0, 0);
                ihi[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, bh, t == 0 ? zi : ihi[j], 0, 0, 0);
            }
        }
        const float dn = h2f((uint32_t)b.hdr[0] & 0xffffu) * kMinPrescale;   // exact: a power of two
        const float *dxs = sm.dx[buf];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            float dxv[16];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 d4 = *reinterpret_cast<const float4 *>(dxs + j * 32 + 8 * i + 4 * lh);
                dxv[4 * i] = d4.x; dxv[4 * i + 1] = d4.y; dxv[4 * i + 2] = d4.z; dxv[4 * i + 3] = d4.w;
            }
#pragma unroll
            for (int v = 0; v < 16; ++v)
                acc[j][v] = fmaf((float)((ihi[j][v] << 3) + ilo[j][v]), dxv[v] * dn, acc[j][v]);
        }
    };

    // a grid with gridDim.y > 1 cuts K: this workgroup does the super-blocks [sb_begin, sb_end) and writes a
    // partial tile that sum_parts_kernel adds to the others in order
    const int64_t sb_begin = nb * blockIdx.y / gridDim.y, sb_end = nb * (blockIdx.y + 1) / gridDim.y;
    load_next(sb_begin);
    store_next((int)(sb_begin & 1));
    __syncthreads();
    for (int64_t sb = sb_begin; sb < sb_end; ++sb) {
        const int buf = (int)(sb & 1);
        DirectB b;   // out of the strip: header of row l%32, then the lane's 64 nibble bytes
        b.hdr = *reinterpret_cast<const v4i *>(park + l32 * 144);
#pragma unroll
        for (int i = 0; i < 4; ++i) b.q[i] = *reinterpret_cast<const v4i *>(park + l32 * 144 + 16 + 64 * lh + 16 * i);
        // past the end the last super-block is fetched again: unconditional loads keep the wait counters exact
        load_next(sb + 1 < sb_end ? sb + 1 : sb_end - 1);
        __builtin_amdgcn_sched_barrier(0);   // the loads stay ahead of the arithmetic they overlap with
        superblock(b, buf);
        store_next(buf ^ 1);
        __syncthreads();
    }

    // ---- store: accumulator register v of lane l is row 8*(v/4) + 4*(l/32) + v%4, column l%32
    const int64_t n = n0 + wave * 32 + l32;
    // the rows' factors (normaliser / 16) go through the idle scale buffer: four rows per read, no load per store
    sm.dx[0][tid & 63] = rs_mine * (1.0f / kMinPrescale);
    __syncthreads();
    // two stretches and no scratch: the output rows were cleared before the launch and both stretches add their
    // tile to them (0 + a + b is a + b in either order, so the result does not depend on which arrives first)
    const bool add = gridDim.y > 1 && part == nullptr;
    float *out = gridDim.y > 1 && !add ? part + (size_t)blockIdx.y * M * N : y;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const float4 f4 = *reinterpret_cast<const float4 *>(&sm.dx[0][j * 32 + 8 * g + 4 * lh]);
            const float f[4] = {f4.x, f4.y, f4.z, f4.w};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t m = m0 + j * 32 + 8 * g + 4 * lh + r;
                if (m < M && n < N) {
                    if (add) unsafeAtomicAdd(out + m * N + n, acc[j][4 * g + r] * f[r]);
                    else out[m * N + n] = acc[j][4 * g + r] * f[r];
                }
            }
        }
    }
}


// ------------------------------------------------------------------------------------------------
// The same product for large batches: every wave keeps its 32 weight rows but works on 128 tokens.
//
// The kernel above spends four vector instructions per matrix instruction on expanding and scaling
// weights, because a converted weight fragment feeds only two token tiles.  Here a wave converts the
// whole super-block of its 32 rows once into 64 registers (both chains, all eight steps) and then
// walks four token tiles with them, so the conversion is paid once per 128 tokens.  Eight waves =
// 256 weight rows x 128 tokens per workgroup, one workgroup per compute unit.
//
// Nothing passes through staging registers: activations, the min-term tile, the activation scales
// and the raw weight blocks go from global memory straight into LDS (global_load_lds, 16 bytes a
// lane, a wave writes one contiguous kilobyte per instruction).  Because such a load cannot pad LDS
// rows, the activation tile is stored [token][256] with the 16-byte segments of a row XOR-swizzled
// by the token index: slot s of token r holds segment s ^ (r & 15), which the loading lane simply
// requests from global memory, and 16 consecutive tokens reading "their" segment g hit 16 different
// slots.
template <int NW>
struct WideSmem {
    int8_t a[2][128 * 256];          // activations of one super-block [token][16 swizzled segments]
    uint16_t ms[2][128 * 16];        // min-term operand [token][8 high | 8 low] (fp16 bits)
    float dx[2][128];                // activation scale of the super-block
    uint8_t park[NW][5 * 1024];      // per wave: raw blocks of its 32 weight rows (4608 bytes used)
};

template <int NW>
__global__ __launch_bounds__(64 * NW, 1) void gemm_q4k_q8k_wide_kernel(const WeightView w, const ActView a, int64_t M,
                                                                      float *__restrict__ y, float *__restrict__ part) {
    static_assert(NW == 8, "the loading roles below are laid out for eight waves");
    constexpr int TM = 128, TN = 32 * NW, JT = TM / 32;
    constexpr int PA = (TM * 16) / (64 * NW);   // 1-KB activation chunks (4 tokens) a wave requests per super-block
    extern __shared__ __align__(16) uint8_t smem_raw[];
    WideSmem<NW> &sm = *reinterpret_cast<WideSmem<NW> *>(smem_raw);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t N = w.N, K = w.K, nb = w.nb;
    int tile_n, tile_m;
    tile_of_workgroup((int)((N + TN - 1) / TN), (int)((M + TM - 1) / TM), tile_n, tile_m);
    const int64_t n0 = (int64_t)tile_n * TN, m0 = (int64_t)tile_m * TM;
    const int l32 = lane & 31, lh = lane >> 5;

    v16f acc[JT];
#pragma unroll
    for (int j = 0; j < JT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[j][v] = 0.f;

    // ---- global -> LDS requests: wave-uniform bases plus 32-bit lane offsets; rows past the edge of
    // a matrix repeat its last valid row (computed, never stored)
    const int64_t wave_row0 = n0 + wave * 32 < N ? n0 + wave * 32 : N - 1;
    const int wrow_cap = (int)(N - 1 - wave_row0 < 31 ? N - 1 - wave_row0 : 31);
    const uint8_t *wbase = w.q4k + wave_row0 * nb * 144;
    uint32_t woff[5];   // piece p = lane + 64*c of the wave's 288 -> row p / 9, 16-byte part p % 9
#pragma unroll
    for (int c = 0; c < 5; ++c) {
        const int p = lane + 64 * c < 287 ? lane + 64 * c : 287;
        const int r = p / 9 < wrow_cap ? p / 9 : wrow_cap;
        woff[c] = (uint32_t)(r * (int)nb * 144 + 16 * (p % 9));
    }
    const int mrow_cap = (int)(M - 1 - m0 < TM - 1 ? M - 1 - m0 : TM - 1);
    const int8_t *abase = a.qs + m0 * K;
    uint32_t aoffg[PA];   // chunk wave + NW*p = tokens 4*chunk .. +3; lane -> token lane/16, slot lane%16
#pragma unroll
    for (int p = 0; p < PA; ++p) {
        const int row = 4 * (wave + NW * p) + (lane >> 4), seg = (lane & 15) ^ (row & 15);
        aoffg[p] = (uint32_t)((row < mrow_cap ? row : mrow_cap) * (int)K + 16 * seg);
    }
    // waves 0..3: min-term tile (2 pieces a token); waves 4, 5: activation scales (one float a token)
    const uint8_t *msbase = reinterpret_cast<const uint8_t *>(a.msum) + m0 * nb * 32;
    const int mstok = (wave & 3) * 32 + (lane >> 1), dxtok = tid & 127;
    const uint32_t msoffg = (uint32_t)((mstok < mrow_cap ? mstok : mrow_cap) * (int)nb * 32 + 16 * (lane & 1));
    const float *dxbase = a.d + m0 * nb;
    const uint32_t dxoffg = (uint32_t)((dxtok < mrow_cap ? dxtok : mrow_cap) * (int)nb);
    // the min-term operand is normalised by the row (rs[m], a power of two): the accumulators run in units of
    // 1 / (16 * rs[m]) until the store, so the activation scales are divided by rs[m] as they are staged (exact)
    const float rs_mine = a.rs[m0 + (dxtok < mrow_cap ? dxtok : mrow_cap)];
    const float inv_rs = 1.0f / rs_mine;
    uint8_t *park = sm.park[wave];

    // Addresses are a scalar base that never moves plus a 32-bit lane offset to which the super-block's
    // displacement is added on the spot: one vector register per request stays live, not a 64-bit pointer.
    const uint8_t *wbase_s = scalar_pointer(wbase);
    const int8_t *abase_s = scalar_pointer(abase);
    const uint8_t *msbase_s = scalar_pointer(msbase);
    const global_ptr<float> dxbase_s = scalar_global(dxbase);
    auto request_strip = [&](uint32_t sb, int c) {
        global_to_lds16(wbase_s + (woff[c] + sb * 144u), park + 1024 * c);
    };
    auto request_act = [&](uint32_t sb, int buf, int p) {
        global_to_lds16(abase_s + (aoffg[p] + sb * 256u), sm.a[buf] + (wave + NW * p) * 1024);
    };
    auto request_ms = [&](uint32_t sb, int buf) {
        if (wave < 4) global_to_lds16(msbase_s + (msoffg + sb * 32u), reinterpret_cast<uint8_t *>(sm.ms[buf]) + wave * 1024);
    };

    // the lane's eight activation reads of a token tile: segment t + 8*(l/32) of token l%32 (+32*j) sits in
    // slot (t + 8*(l/32)) ^ (l%16) = t ^ z with z = 8*(l/32) ^ (l%16), i.e. at byte (256*(l%32) + 16*z) ^ 16*t
    const int aoffl = l32 * 256 + 16 * ((8 * lh) ^ (l32 & 15));
    const v16i zi = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

    // both scaled int8 copies of the lane's 128 weights (step t = sub-block 4*(l/32) + t/2, half t%2) and the header
    v4i hdr, cl[8], ch[8];
    uint32_t lo_w, hi_w;   // base-8 digits of the lane's four sub-block scales
    auto read_header = [&]() {
        hdr = *reinterpret_cast<const v4i *>(park + l32 * 144);
        const ScalesK4 sc = unpack_scales_k4((uint32_t)hdr[1], (uint32_t)hdr[2], (uint32_t)hdr[3]);
        const uint32_t scw = lh ? sc.sc_hi : sc.sc_lo;
        lo_w = scw & 0x07070707u;
        hi_w = (scw >> 3) & 0x07070707u;
    };
    auto strip_piece = [&](int t) {   // nibble bytes of step t: 16-byte piece 2*(t/4) + t%2 of the lane's 64
        return *reinterpret_cast<const v4i *>(park + l32 * 144 + 16 + 64 * lh + 16 * (2 * (t >> 2) + (t & 1)));
    };
    auto convert = [&](int t, const v4i &raw) {
        const int i = t >> 1, nib = i & 1;
        const uint32_t sl = byte_to_u16x2(lo_w, i), sh = byte_to_u16x2(hi_w, i);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t x = nib ? ((uint32_t)raw[c] >> 4) & 0x0f0f0f0fu : (uint32_t)raw[c] & 0x0f0f0f0fu;
            cl[t][c] = (int)pk_mul_u16(x, sl);
            ch[t][c] = (int)pk_mul_u16(x, sh);
        }
    };

    // a grid with gridDim.y > 1 cuts K: this workgroup does the super-blocks [sb_begin, sb_end) and writes a
    // partial tile that sum_parts_kernel adds to the others in order
    const int64_t sb_begin = nb * blockIdx.y / gridDim.y, sb_end = nb * (blockIdx.y + 1) / gridDim.y;
    // ---- prologue: requests of the first super-block
#pragma unroll
    for (int c = 0; c < 5; ++c) request_strip((uint32_t)sb_begin, c);
#pragma unroll
    for (int p = 0; p < PA; ++p) request_act((uint32_t)sb_begin, 0, p);
    request_ms((uint32_t)sb_begin, 0);
    sm.dx[0][tid & 127] = dxbase_s[dxoffg + (uint32_t)sb_begin] * inv_rs;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();

    // The two waves that share a SIMD (w and w+4) must not want the same pipe at the same time: the older one
    // wins every arbitration and the younger one only gets what is left.  So they run the same super-block in
    // opposite orders.  EARLY waves (0..3) convert the weights of a super-block at its start (vector work first,
    // the conversion of step t+1 sits between the matrix instructions of step t of the first tile); LATE waves
    // (4..7) convert the weights of the NEXT super-block at the end of the current one, after their last tile,
    // so that they start every super-block with matrix work while their partner converts.
    //
    // Inside a super-block the order is pinned step by step (the scheduling barriers let nothing cross): four
    // activation fragments are always in flight, a fragment register is refilled as soon as its two matrix
    // instructions are issued, the activation scales of a tile arrive two groups at a time ahead of its flush, the next
    // tile's first fragments while its integer sums are put together.  The requests for the next super-block are issued one per step
    // in the tiles without conversion work: all waves asking at once right after the barrier only queue up in
    // the memory pipeline.
    auto run = [&](auto late_tag) {
        constexpr bool LATE = decltype(late_tag)::value;
        if (LATE) {   // weights of the first super-block, with nothing to overlap
            read_header();
#pragma unroll
            for (int t = 0; t < 8; ++t) convert(t, strip_piece(t));
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the strip is about to be overwritten
        }
        for (int64_t sb = sb_begin; sb < sb_end; ++sb) {
            const int buf = (int)((sb - sb_begin) & 1);
            const uint32_t sb_next = (uint32_t)(sb + 1 < sb_end ? sb + 1 : sb_end - 1);   // past the end: requested again, never used
            v4i raw[4];
            if (!LATE) {   // out of the strip: header of row l%32, then the lane's 64 nibble bytes
                read_header();
#pragma unroll
                for (int i = 0; i < 4; ++i) raw[i] = *reinterpret_cast<const v4i *>(park + l32 * 144 + 16 + 64 * lh + 16 * i);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the strip is about to be overwritten
            }
            const float dxreg = dxbase_s[dxoffg + sb_next];
            __builtin_amdgcn_sched_barrier(0);
            const int8_t *ab = sm.a[buf];
            const uint8_t *msb = reinterpret_cast<const uint8_t *>(sm.ms[buf]);
            const float *dxs = sm.dx[buf];
            auto fragment = [&](int j, int t) {
                return *reinterpret_cast<const v4i *>(ab + j * 32 * 256 + (aoffl ^ (16 * t)));
            };
            v4i ring[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) ring[t] = fragment(0, t);
            // ---- min term: -dmin*min of the 8 sub-blocks as fp16 high and low parts
            const float dn = h2f((uint32_t)hdr[0] & 0xffffu) * kMinPrescale;   // exact: a power of two
            {
                const ScalesK4 sc = unpack_scales_k4((uint32_t)hdr[1], (uint32_t)hdr[2], (uint32_t)hdr[3]);
                const float ndmin = -h2f((uint32_t)hdr[0] >> 16);
                v8h mh, ml;
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    _Float16 h, l;
                    split_h(ndmin * (float)min_k4(sc, t), h, l);
                    mh[t] = h;
                    ml[t] = lh ? (_Float16)0.f : l;
                }
#pragma unroll
                for (int j = 0; j < JT; ++j) {
                    const v8h am = *reinterpret_cast<const v8h *>(msb + (j * 32 + l32) * 32 + 16 * lh);
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(am, mh, acc[j], 0, 0, 0);
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(am, ml, acc[j], 0, 0, 0);
                }
            }
            if (!LATE) convert(0, raw[0]);
            __builtin_amdgcn_sched_barrier(0);
            // A finished tile's chains become one integer sum an output right away; the rest of its flush goes between the matrix
            // instructions of the next tile, two outputs a step (the last tile's follows it).  The whole flush behind every
            // tile: 4096 -> 2 x 14336 at 512 tokens 160.0 -> 155.6 us, at 1024 303.6 -> 298.5.
            v16i whole;
            v4i dq[2];
            auto read_dq = [&](int j, int i) { dq[i & 1] = *reinterpret_cast<const v4i *>(dxs + j * 32 + 8 * i + 4 * lh); };
            auto flush_two = [&](int j, int t) {
#pragma unroll
                for (int v = 2 * t; v < 2 * t + 2; ++v) {
                    acc[j][v] = fmaf((float)whole[v], __int_as_float(dq[(v >> 2) & 1][v & 3]) * dn, acc[j][v]);
                    asm volatile("" : "+v"(acc[j][v]));
                }
            };
#pragma unroll
            for (int j = 0; j < JT; ++j) {
                v16i ilo, ihi;
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    ilo = __builtin_amdgcn_mfma_i32_32x32x32_i8(ring[t & 3], cl[t], t == 0 ? zi : ilo, 0, 0, 0);
                    ihi = __builtin_amdgcn_mfma_i32_32x32x32_i8(ring[t & 3], ch[t], t == 0 ? zi : ihi, 0, 0, 0);
                    if (t < 4) ring[t & 3] = fragment(j, t + 4);
                    if (j > 0) {
                        flush_two(j - 1, t);
                        if (t & 1) { if (t < 5) read_dq(j - 1, (t >> 1) + 2); }
                    }
                    if (t >= 6) read_dq(j, t - 6);
                    if (!LATE && j == 0 && t < 7) convert(t + 1, raw[2 * ((t + 1) >> 2) + ((t + 1) & 1)]);
                    // requests for the next super-block, one per step: the strip first (its previous content was
                    // read at the top of this trip by the early waves, at the end of the last one by the late waves)
                    if (j == (LATE ? 0 : 1) && t < 5) request_strip(sb_next, t);
                    if (j == (LATE ? 1 : 2) && (t & 1)) request_act(sb_next, buf ^ 1, t >> 1);
                    if (j == (LATE ? 1 : 2) && t == 0) request_ms(sb_next, buf ^ 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (j + 1 < JT) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) ring[t] = fragment(j + 1, t);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int v = 0; v < 16; ++v) whole[v] = (ihi[v] << 3) + ilo[v];
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                flush_two(JT - 1, t);
                if ((t & 1) && t < 5) read_dq(JT - 1, (t >> 1) + 2);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (LATE) {
                // the next super-block's raw weights were requested at the top of this trip; of the requests
                // made since then (four activation chunks; these waves load no min-term piece) none needs
                // to have landed
                asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
                read_header();
#pragma unroll
                for (int t = 0; t < 8; ++t) convert(t, strip_piece(t));
            }
            sm.dx[buf ^ 1][tid & 127] = dxreg * inv_rs;   // every thread stores (a repeated value past 128): no branch
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __syncthreads();
        }
    };
    if (wave < 4) run(std::false_type{});
    else run(std::true_type{});

    // ---- store: accumulator register v of lane l is row 8*(v/4) + 4*(l/32) + v%4, column l%32
    const int64_t n = n0 + wave * 32 + l32;
    // the rows' factors (normaliser / 16) go through the idle scale buffer: four rows per read, no load per store
    sm.dx[0][tid & 127] = rs_mine * (1.0f / kMinPrescale);
    __syncthreads();
    // two stretches and no scratch: the output rows were cleared before the launch and both stretches add their
    // tile to them (0 + a + b is a + b in either order, so the result does not depend on which arrives first)
    const bool add = gridDim.y > 1 && part == nullptr;
    float *out = gridDim.y > 1 && !add ? part + (size_t)blockIdx.y * M * N : y;
#pragma unroll
    for (int j = 0; j < JT; ++j) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const float4 f4 = *reinterpret_cast<const float4 *>(&sm.dx[0][j * 32 + 8 * g + 4 * lh]);
            const float f[4] = {f4.x, f4.y, f4.z, f4.w};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t m = m0 + j * 32 + 8 * g + 4 * lh + r;
                if (m < M && n < N) {
                    if (add) unsafeAtomicAdd(out + m * N + n, acc[j][4 * g + r] * f[r]);
                    else out[m * N + n] = acc[j][4 * g + r] * f[r];
                }
            }
        }
    }
}

}  // namespace

namespace {
// n matrices of one type and K over the same rows.  A launch takes as many of them as have room for their partial
// tiles in the scratch; the next launch uses the same bytes again, behind the adding passes.
template <int QT>
hipError_t launch_per32(int n, const WeightView *w, const ActView &a, int64_t M, float *const *y, const Scratch &sc, hipStream_t s) {
    if (n < 1 || n > kMaxTargets || w[0].K > (1 << 24)) return hipErrorInvalidValue;   // 32-bit lane offsets: 128 rows of K bytes
    const auto kern = &gemm_per32_kernel<QT>;
    if (!dry_run()) {
        static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(GemmSmem));
        if (attr != hipSuccess) return attr;
    }
    for (int first = 0; first < n;) {
        Per32Args g{};
        g.a = a;
        g.M = M;
        SumTargets sums{};
        size_t used = 0;
        int64_t wg = 0;
        int i = first;
        for (; i < n; ++i) {
            if (w[i].K != w[0].K) return hipErrorInvalidValue;
            const int n_split = sc.p ? per32_splits(QT, w[i].K, M, w[i].N) : 1;
            const size_t bytes = n_split > 1 ? (size_t)n_split * M * w[i].N * 4 : 0;
            if (used + bytes > sc.bytes && bytes) {
                if (i == first) return hipErrorInvalidValue;   // partial tiles would not fit
                break;
            }
            const int64_t tiles = per32_tiles(M, w[i].N), pad = (tiles + 7) / 8 * 8;
            if (wg + pad * n_split >= 0x7fffffff) {
                if (i == first) return hipErrorInvalidValue;
                break;
            }
            Per32Target &t = g.t[g.n++];
            t.w = w[i];
            t.out = y[i];
            if (bytes) {
                if (!dry_run()) t.out = sc.p + used / 4;
                add_sum(sums, t.out, y[i], n_split, M * w[i].N);
                used += bytes;
            }
            t.tiles_pad = (int)pad;
            t.n_split = n_split;
            t.first_wg = (int)wg;
            wg += pad * n_split;
            if (dry_run())
                plan_note("gemm_per32_kernel<%s>%s: tile 128 tokens x 128 rows, %lld tiles x %d K stretches%s", plan_type_name(QT),
                          g.n > 1 ? " (same launch)" : "", (long long)tiles, n_split, n_split > 1 ? " + sum_parts_kernel" : "");
        }
        first = i;
        if (dry_run()) {
            if (sums.n) plan_note_cut();
            continue;
        }
        hipLaunchKernelGGL(kern, dim3((unsigned)wg), dim3(kGemmThreads), sizeof(GemmSmem), s, g);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess && sums.n) e = launch_sum_parts(sums, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
}  // namespace

hipError_t launch_sum_parts(const float *part, int n_split, size_t n, float *y, hipStream_t s) {
    if (dry_run()) {
        plan_note("sum_parts_kernel: adds %d partial results of %zu outputs in order", n_split, n);
        return hipSuccess;
    }
    SumTargets g{};
    add_sum(g, part, y, n_split, (int64_t)n);   // callers only split when n is a multiple of 4
    return launch_sum_parts(g, s);
}

// (The figures at 33 .. 256 tokens below were taken when those batches came here; most of them stream now, stream_takes.)
// K stretches for the kernels that take ggml-format activations (64-token x 128-row tiles, two workgroups per
// compute unit = 512 places): below 384 tiles K is cut in 2, below 192 in 3, below 96 in 4, below 64 in 8, never under twelve super-blocks a
// stretch (K = 4096 cut in two measured slower than whole: the pass that adds the partial tiles costs more
// than the fuller grid gains).
int q8k_tile_splits(int64_t K, int64_t M, int64_t N, bool add_ok) {
    static const int forced = tuning_int("QPROJ_Q8K_SPLITS", 0);
    static const bool no_add = tuning_int("QPROJ_NO_TILE_ADD", 0) != 0;
    const int64_t tiles = ((N + 127) / 128) * ((M + 63) / 64);
    // Two stretches that add themselves to cleared output rows cost no pass over partial tiles: from 96 tiles on that
    // beats three stretches with the pass, and K = 4096 (eight super-blocks a stretch) is worth cutting while the whole-K
    // tiles would not give every compute unit a workgroup.  Per call, us: 4096 x 4096 at 192 / 256 tokens 32.7 / 34.2 ->
    // 26.5 / 28.8 (at 512 tokens, 256 tiles, the cut loses: 39.9 -> 42.8, so it stays whole); 4096 -> 14336 at 64 tokens
    // 32.0 -> 27.7; 14336 -> 4096 at 192 / 256 tokens 65.3 / 67.6 -> 59.9 / 63.2.
    if (add_ok && !no_add && forced <= 0 && (M * N) % 4 == 0 && tiles >= 96 && tiles < 384 && K / 256 >= 16 &&
        (K / 256 >= 24 || tiles < 256))
        return 2;
    // (under 64 tiles - a down projection of 4096 rows at up to 64 tokens is 32 - eight stretches: 14336 -> 4096 at
    // 33 / 64 tokens, four -> eight stretches, Q6_K 42.0 / 43.5 -> 29.7 / 31.1 us, Q4_K 35.6 / 37.4 -> 27.9 / 29.7; ten to
    // fourteen were slower again, the pass over the partial tiles grows; 64 tiles keep four: seven 47.2 -> 46.1 for Q6_K
    // and 40.5 -> 42.8 for Q4_K)
    int n = forced > 0 ? forced : tiles >= 384 ? 1 : tiles >= 192 ? 2 : tiles >= 96 ? 3 : tiles >= 64 ? 4 : 8;
    if ((M * N) % 4 != 0) n = 1;
    // a stretch is at least 12 super-blocks (the pass that adds the partial tiles has to be earned), 4 where the
    // grid is under a fifth of the workgroups the chip holds and a workgroup's K loop is pure latency
    const int min_sb = tiles >= 192 ? 12 : 4;
    while (n > 1 && K / 256 < min_sb * n) --n;
    return n;
}
size_t q8k_tile_scratch_bytes(int64_t K, int64_t M, int64_t N) {
    const int n = q8k_tile_splits(K, M, N, false);
    return n > 1 ? (size_t)n * M * N * 4 : 0;
}

// A grid of fewer than 192 tiles leaves the 256 compute units mostly idle and a workgroup's K loop is
// latency-bound: K is then cut into stretches done by different workgroups, as many as fill one round (32 tiles of
// K = 14336, Q8_0 at 64 - 128 tokens: 8 stretches instead of 3).  The cut follows the matrix and the row count alone,
// whatever shares the launch: the order of a result's fp32 sums is the same in a call of its own, and the shorter
// chains keep the error down (8192 -> 8192 / 1024 / 1024 at 256 rows against 64 bits: 2.1e-7; with the cut by the tiles of
// the whole launch, which was tried, 2.9e-7).
int64_t per32_tiles(int64_t M, int64_t N) { return ((N + BN - 1) / BN) * ((M + BM - 1) / BM); }
int per32_splits(int type, int64_t K, int64_t M, int64_t N) {
    static const int forced = tuning_int("QPROJ_PER32_SPLITS", 0);
    // as many stretches as fill one round of workgroups (one a compute unit), eight at most
    const int64_t tiles = per32_tiles(M, N);
    int n = forced > 0 ? forced : tiles >= 192 ? 1 : (int)std::min<int64_t>(8, std::max<int64_t>(1, cu_count() / tiles));
    if ((M * N) % 4 != 0) n = 1;
    // at least two times 256 weights a stretch, Q4_K four (its min term is a loop of its own over the stretch).  Q8_0,
    // four -> two, us: 4096 -> 1024 at 64 tokens 21.2 -> 16.8, 2560 x 2560 at 250 27.2 -> 22.5, 4096 x 4096 at 100 24.5 -> 22.4.
    const int least = type == kTypeQ8_0 ? 2 : 4;
    while (n > 1 && K / 256 < least * n) --n;
    // no stretch without work: 12 times 256 weights in five stretches of three leave the fifth empty (the same sums with four)
    const int64_t units = (K + 255) / 256;
    while (n > 1 && (units + n - 2) / (n - 1) == (units + n - 1) / n) --n;
    return n;
}
size_t per32_scratch_bytes(int type, int64_t K, int64_t M, int64_t N) {
    if (type == kTypeQ8_0 && q8_0_tokens_takes(K, M, N)) return q8_0_tokens_scratch_bytes(K, M, N);
    const int n = per32_splits(type, K, M, N);
    return n > 1 ? (size_t)n * M * N * 4 : 0;
}

hipError_t launch_gemm_q8x32(const WeightView &w, const ActView &a, int64_t M, float *y, const Scratch &scratch, hipStream_t s) {
    if (w.type != kTypeQ4_K || w.K % 256 != 0 || M <= 0 || !a.msum || !a.rs) return hipErrorInvalidValue;
    return launch_per32<kTypeQ4_K>(1, &w, a, M, &y, scratch, s);
}

// Q8_0 weights x ggml Q8_0 activation blocks (planes in `a`), K a multiple of 128
hipError_t launch_gemm_q8_0(int n, const WeightView *w, const ActView &a, int64_t M, float *const *y, const Scratch &scratch, hipStream_t s) {
    WeightView tokens[kMaxTargets], tiled[kMaxTargets];
    float *yt[kMaxTargets], *yl[kMaxTargets];
    int nt = 0, nl = 0;
    if (n < 1 || n > kMaxTargets) return hipErrorInvalidValue;
    for (int i = 0; i < n; ++i) {
        if (w[i].type != kTypeQ8_0 || a.kind != kActKindQ8_0 || w[i].K % BK != 0 || M <= 0) return hipErrorInvalidValue;
        if (q8_0_tokens_takes(w[i].K, M, w[i].N)) {
            tokens[nt] = w[i];
            yt[nt++] = y[i];
        } else {
            tiled[nl] = w[i];
            yl[nl++] = y[i];
        }
    }
    if (nt) {
        const hipError_t e = launch_gemm_q8_0_tokens(nt, tokens, a, M, yt, scratch, s);
        if (e != hipSuccess) return e;
    }
    return nl ? launch_per32<kTypeQ8_0>(nl, tiled, a, M, yl, scratch, s) : hipSuccess;
}

// Which Q4_K kernel and how many stretches of K (one rule for the launcher and for the scratch sizing).  The
// 128-token kernel (256 weight rows a workgroup, one workgroup per compute unit) wants about 192 workgroups or more:
// a grid of 48..191 such tiles is multiplied by cutting K into the stretches wide_tile_splits picks (64 tiles of
// K = 14336: four; of K = 11008: three, 192 workgroups, where the halving rule before left half the chip idle).
// Everything else takes 64-token tiles with the stretches of q8k_tile_splits.
namespace {
struct Q4Plan {
    bool wide;
    int n_split;
};
// add_ok: the output rows hold zeros when the launch starts (Scratch::zeroed)
Q4Plan q4k_plan(int64_t K, int64_t M, int64_t N, bool have_scratch, bool add_ok = false) {
    static const int wide_env = tuning_int("QPROJ_Q8K_WIDE", -1);
    const int64_t wide_tiles = ((N + 255) / 256) * ((M + 127) / 128);
    if (wide_env >= 0 ? wide_env != 0 : wide_tiles >= 192) return {true, 1};
    if (wide_env < 0 && have_scratch && (M * N) % 4 == 0 && wide_tiles >= 48) {
        const int n = wide_tile_splits(wide_tiles, K / 256, M, N, cu_count(), 4.5);
        if (n > 1) return {true, n};
    }
    return {false, have_scratch || add_ok ? q8k_tile_splits(K, M, N, add_ok) : 1};
}
}  // namespace


bool q4k_fills_wide(int64_t K, int64_t M, int64_t N) {
    const Q4Plan p = q4k_plan(K, M, N, true);
    return p.wide && ((N + 255) / 256) * ((M + 127) / 128) * p.n_split * 8 >= (int64_t)cu_count() * 5;
}

size_t q4k_tile_scratch_bytes(int64_t K, int64_t M, int64_t N) {
    const Q4Plan p = q4k_plan(K, M, N, true);
    return p.n_split > 1 ? (size_t)p.n_split * M * N * 4 : 0;
}

// ggml-format activations (Q8_K planes in `a`, including the min-term plane), Q4_K weights, any M
hipError_t launch_gemm_q8k(const WeightView &w, const ActView &a, int64_t M, float *y, const Scratch &scratch, hipStream_t s) {
    if (w.type != kTypeQ4_K || a.kind != kActKindQ8_K || !a.msum || !a.rs || M <= 0) return hipErrorInvalidValue;
    if (w.K > (1 << 24)) return hipErrorInvalidValue;   // 32-bit lane offsets: 128 token rows of K bytes, 32 weight rows of K*144/256
    const bool zeroed = (scratch.zeroed & 1u) != 0;
    Q4Plan p = q4k_plan(w.K, M, w.N, scratch.p != nullptr, zeroed);
    const bool add = zeroed && p.n_split == 2;   // both stretches add to the cleared rows: no partial tiles
    if (zeroed && !add) p = q4k_plan(w.K, M, w.N, scratch.p != nullptr);
    if (p.n_split > 1 && !add && (size_t)p.n_split * M * w.N * 4 > scratch.bytes) return hipErrorInvalidValue;   // partial tiles would not fit
    if (dry_run()) {
        if (p.n_split > 1 && !add) plan_note_cut();
        const long long tiles = p.wide ? (long long)(((w.N + 255) / 256) * ((M + 127) / 128)) : (long long)(((w.N + 127) / 128) * ((M + 63) / 64));
        plan_note("%s: tile %s, %lld tiles x %d K stretches%s, partial tiles %zu B", p.wide ? "gemm_q4k_q8k_wide_kernel" : "gemm_q4k_q8k_direct_kernel",
                  p.wide ? "128 tokens x 256 rows" : "64 tokens x 128 rows", tiles, p.n_split,
                  p.n_split == 1 ? "" : add ? ", the two stretches add themselves to cleared rows" : " + sum_parts_kernel",
                  p.n_split > 1 && !add ? (size_t)p.n_split * M * w.N * 4 : (size_t)0);
        return hipSuccess;
    }
    float *const part = add ? nullptr : scratch.p;
    if (p.wide) {   // 128 tokens x 256 weight rows per workgroup, one workgroup per compute unit
        using Smem = WideSmem<8>;
        const auto kern = &gemm_q4k_q8k_wide_kernel<8>;
        static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(Smem));
        if (attr != hipSuccess) return attr;
        const int64_t wide_tiles = ((w.N + 255) / 256) * ((M + 127) / 128);
        hipLaunchKernelGGL(kern, dim3((unsigned)wide_tiles, (unsigned)p.n_split), dim3(512), sizeof(Smem), s, w, a, M, y, part);
        if (p.n_split > 1 && !add) return launch_sum_parts(scratch.p, p.n_split, (size_t)M * w.N, y, s);
        return hipGetLastError();
    }
    constexpr int NW = 4;   // 64 tokens x 128 weight rows per workgroup, two workgroups per compute unit
    using Smem = DirectSmem<NW>;
    static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_q4k_q8k_direct_kernel<NW>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(Smem));
    if (attr != hipSuccess) return attr;
    const dim3 grid((unsigned)(((w.N + 32 * NW - 1) / (32 * NW)) * ((M + 63) / 64)), (unsigned)p.n_split);
    DirectTargets tg{};
    tg.n = 1;
    tg.w[0] = w;
    tg.y[0] = y;
    hipLaunchKernelGGL(gemm_q4k_q8k_direct_kernel<NW>, grid, dim3(64 * NW), sizeof(Smem), s, tg, a, M, part);
    if (p.n_split > 1 && !add) return launch_sum_parts(scratch.p, p.n_split, (size_t)M * w.N, y, s);
    return hipGetLastError();
}

namespace {
// Which of n matrices over the same activation rows share ONE launch of the 64-token kernel: those that would take it
// with K in one stretch (or are small enough to be better off together than cut).  The others (128-token tiles, K cut
// into stretches) get launches of their own.  Fills joined[], returns how many (0 or >= 2).
int q4k_joined_set(int n, const WeightView *w, int64_t M, bool have_scratch, bool planes_ok, int (&joined)[3]) {
    static const int wide_env = tuning_int("QPROJ_Q8K_WIDE", -1);
    static const bool off = tuning_int("QPROJ_Q8K_NO_MULTI", 0) != 0;
    const bool can = !off && n >= 2 && n <= 3 && wide_env < 0 && planes_ok && M > 0;
    int n_joined = 0;
    for (int i = 0; i < n; ++i) {
        const Q4Plan p = q4k_plan(w[i].K, M, w[i].N, have_scratch);
        const bool fits = can && w[i].type == kTypeQ4_K && w[i].K == w[0].K && w[i].K <= (1 << 24) && !p.wide &&
                          (p.n_split == 1 || ((w[i].N + 127) / 128) * ((M + 63) / 64) < 96);   // small ones are better off together than cut
        if (fits) joined[n_joined++] = i;
    }
    return n_joined < 2 ? 0 : n_joined;
}
}  // namespace

// bit i: matrix i of a launch_gemm_q8k_multi call gets a launch of its own that cuts K in two stretches which add
// themselves, if its output rows are cleared beforehand
uint32_t q4k_multi_adds(int n, const WeightView *w, int64_t M, bool have_scratch) {
    int joined[3];
    const int n_joined = n <= 3 ? q4k_joined_set(n, w, M, have_scratch, true, joined) : 0;
    uint32_t mask = 0;
    for (int i = 0; i < n; ++i) {
        bool in = false;
        for (int j = 0; j < n_joined; ++j) in = in || joined[j] == i;
        if (!in && w[i].type == kTypeQ4_K && q4k_plan(w[i].K, M, w[i].N, have_scratch, true).n_split == 2) mask |= 1u << i;
    }
    return mask;
}

// The same for n matrices over the same activation rows.  One launch where every matrix would take the
// 64-token kernel with K in one stretch; otherwise one launch a matrix, as above.
hipError_t launch_gemm_q8k_multi(int n, const WeightView *w, const ActView &a, int64_t M, float *const *y,
                                 const Scratch &scratch, hipStream_t s) {
    constexpr int NW = 4;
    int joined[3];
    int n_joined = n <= 3 ? q4k_joined_set(n, w, M, scratch.p != nullptr, a.kind == kActKindQ8_K && a.msum && a.rs, joined) : 0;
    for (int i = 0; i < n; ++i) {
        bool in = false;
        for (int j = 0; j < n_joined; ++j) in = in || joined[j] == i;
        if (in) continue;
        hipError_t e = launch_gemm_q8k(w[i], a, M, y[i], scratch.for_target(i), s);
        if (e != hipSuccess) return e;
    }
    if (n_joined == 0) return hipSuccess;
    if (dry_run()) {
        long long wgs = 0;
        for (int j = 0; j < n_joined; ++j) {
            wgs += (long long)(((w[joined[j]].N + 32 * NW - 1) / (32 * NW)) * ((M + 63) / 64));
            wgs = (wgs + 7) / 8 * 8;
        }
        plan_note("gemm_q4k_q8k_direct_kernel: %d matrices in one launch, tile 64 tokens x 128 rows, %lld workgroups, K whole", n_joined, wgs);
        return hipSuccess;
    }
    using Smem = DirectSmem<NW>;
    static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_q4k_q8k_direct_kernel<NW>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(Smem));
    if (attr != hipSuccess) return attr;
    DirectTargets tg{};
    tg.n = n_joined;
    int64_t wg = 0;
    for (int j = 0; j < n_joined; ++j) {
        const int i = joined[j];
        tg.w[j] = w[i];
        tg.y[j] = y[i];
        tg.first_wg[j] = (int)wg;
        wg += ((w[i].N + 32 * NW - 1) / (32 * NW)) * ((M + 63) / 64);
        wg = (wg + 7) / 8 * 8;   // the next matrix starts on XCD 0 again
    }
    if (wg >= 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL(gemm_q4k_q8k_direct_kernel<NW>, dim3((unsigned)wg), dim3(64 * NW), sizeof(Smem), s, tg, a, M,
                       static_cast<float *>(nullptr));
    return hipGetLastError();
}

}  // namespace qproj
