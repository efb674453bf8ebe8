// Raw K-quant blocks -> int8 matrix-core operands, shared by the tiled kernels (gfx950).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "qproj_device.h"

namespace qproj {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef unsigned short v2us __attribute__((ext_vector_type(2)));

// waits until at most N of the wave's vector memory requests (global -> LDS ones among them) are outstanding
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ uint32_t pk_mul_u16(uint32_t x, uint32_t s2) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2us, x) * __builtin_bit_cast(v2us, s2));
}

__device__ __forceinline__ uint32_t byte_to_u16x2(uint32_t word, int i) {
    // byte i of word -> both 16-bit halves (v_perm_b32: selector 0x0c yields a zero byte)
    return __builtin_amdgcn_perm(0u, word, 0x0c000c00u | (uint32_t)(i << 16) | (uint32_t)i);
}

// eight bytes below 128 -> exact fp16 integers: 0x6400 | b is 1024 + b
__device__ __forceinline__ v8h bytes_to_f16(uint32_t b0123, uint32_t b4567) {
    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
    const v2h k = {(_Float16)1024.f, (_Float16)1024.f};
    v8h r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t w = i < 2 ? b0123 : b4567;
        const uint32_t p = __builtin_amdgcn_perm(0x64646464u, w, (i & 1) ? 0x04030402u : 0x04010400u);
        const v2h h = __builtin_bit_cast(v2h, p) - k;
        r[2 * i] = h[0];
        r[2 * i + 1] = h[1];
    }
    return r;
}

// 16 nibbles of a Q4_K sub-block (low ones for even i) times both base-8 digits of its scale; byte i of lo_w / hi_w
__device__ __forceinline__ void convert_q4k(const v4i &raw, uint32_t lo_w, uint32_t hi_w, int i, v4i &cl, v4i &ch) {
    const uint32_t sl = byte_to_u16x2(lo_w, i), sh = byte_to_u16x2(hi_w, i);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const uint32_t x = (i & 1) ? ((uint32_t)raw[c] >> 4) & 0x0f0f0f0fu : (uint32_t)raw[c] & 0x0f0f0f0fu;
        cl[c] = (int)pk_mul_u16(x, sl);
        ch[c] = (int)pk_mul_u16(x, sh);
    }
}

// two 16-bit lanes: x * s + c, each lane modulo 2^16
__device__ __forceinline__ uint32_t pk_mad_u16(uint32_t x, uint32_t s, uint32_t c) {
    uint32_t r;
    asm("v_pk_mad_u16 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(s), "v"(c));
    return r;
}

// The 16 + 16 weights that one 16-byte piece of ql (group gl of the half, bytes 16e .. 16e+15) holds in its low and
// high nibbles, with the matching piece of qh, into both int8 operands.  Step t of a lane is sub-block 8f + t of its
// half f = group g = t/2 (ql byte 32*(g%2) + l, nibble g/2, qh bits 2g and 2g+1), bytes l = 16*(t%2) .. +15; `scq`
// holds the eight scales of the half.
__device__ __forceinline__ void convert_q6k(const v4i &lq, const v4i &hq, const v2i &scq, int gl, int e, v4i (&cl)[8], v4i (&ch)[8]) {
#pragma unroll
    for (int nib = 0; nib < 2; ++nib) {
        const int g = gl + 2 * nib, t = 2 * g + e;
        const int s = (int)(int8_t)((uint32_t)scq[t >> 2] >> (8 * (t & 3)));
        const uint32_t s16 = __builtin_amdgcn_perm((uint32_t)s, (uint32_t)s, 0x01000100u);
        const int cc = 128 - 32 * s;
        const uint32_t c16 = __builtin_amdgcn_perm((uint32_t)cc, (uint32_t)cc, 0x01000100u);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t lw = (uint32_t)lq[c], hw = (uint32_t)hq[c];
            const uint32_t x = nib ? (lw >> 4) & 0x0f0f0f0fu : lw & 0x0f0f0f0fu;
            const uint32_t hs = g == 0 ? hw << 4 : g == 1 ? hw << 2 : g == 2 ? hw : hw >> 2;
            const uint32_t q = (hs & 0x30303030u) | x;                          // four codes 0..63
            // codes 0, 2 and 1, 3 in 16-bit lanes: byte permutes over zeros (a mask for the first pair made the compiler
            // build the four codes twice, once for each pair)
            const uint32_t e0 = __builtin_amdgcn_perm(0u, q, 0x0c020c00u), e1 = __builtin_amdgcn_perm(0u, q, 0x0c030c01u);
            const uint32_t w0 = pk_mad_u16(e0, s16, c16), w1 = pk_mad_u16(e1, s16, c16);   // sc * (q - 32) + 128
            // low bytes (bit 7 flipped: minus 128 modulo 256) and high bytes, back in the order of the codes
            cl[t][c] = (int)(__builtin_amdgcn_perm(w1, w0, 0x06020400u) ^ 0x80808080u);
            ch[t][c] = (int)__builtin_amdgcn_perm(w1, w0, 0x07030501u);
        }
    }
}

}  // namespace qproj
