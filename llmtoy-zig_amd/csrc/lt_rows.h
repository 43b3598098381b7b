// lt_rows.h -- the work units of Q8_0, Q4_K and Q6_K rows against fp32
// activations held in registers: shared by the matvec (lt_matvec.hip) and
// the expert kernels by id (lt_q4k.hip), which keep a thread at one unit
// position and walk the rows.
#pragma once

#include "lt_internal.h"
#include "lt_limbs.h"

namespace lt {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

// acc + (low, high f16 of the word) * (x0, x1), fp32: v_fma_mix_f32 reads the
// f16 operand in place.  A code q in the low bits of a half word is the f16
// subnormal q 2^-24, exact in the product, so no code is converted: the sums
// carry 2^-24, which the block scale takes back (exactly).
__device__ __forceinline__ float fma_codes(uint32_t w, float x0, float x1, float acc) {
    const half2_t h = __builtin_bit_cast(half2_t, w);
    return fmaf((float)h[1], x1, fmaf((float)h[0], x0, acc));
}

// The n / 4 quads of a unit's activations, quad t at p[t * stride].
__device__ __forceinline__ void load_x(const float4 *p, int stride, float *v, int n) {
#pragma unroll
    for (int t = 0; t < n / 4; t++) {
        const float4 f = p[t * stride];
        v[4 * t] = f.x; v[4 * t + 1] = f.y; v[4 * t + 2] = f.z; v[4 * t + 3] = f.w;
    }
}

__device__ __forceinline__ float sum16(const float *v) {
    const float a = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    const float b = ((v[8] + v[9]) + (v[10] + v[11])) + ((v[12] + v[13]) + (v[14] + v[15]));
    return a + b;
}

// ---- formats: elements per unit (kElems), the unit and quad within it of
// activations 4 f + [0, 4), the unit's activations from its quads, the loads
// of unit i behind unit u0 of the matrix, and the unit's dot product.  For the
// matvec's launch shapes (lt_matvec.hip): load buffers in runs of many passes
// (ND), the wavefronts that a CU holds with one buffer (waves: the registers
// allow 32 for Q8_0, but rows of more than 256 units take as much LDS for x
// that fewer are better), the numbers of buffers to choose from (takes), and
// the constants of its estimate.
struct FmtQ8_0 {
    static constexpr int kElems = 32, ND = 4;
    static constexpr double kRound = 0.85, kLanes = 1536, kKeep = 0.85, kLong = 1e9;
    static int waves(int U) { return U <= 256 ? 32 : 16; }
    static bool takes(int U, int nd, bool runs) { return (nd > 1) == (runs && U > 256); }
    struct X {
        float v[32];
    };
    struct Regs {
        uint4 q0, q1;
        uint16_t d;
    };
    static __device__ __forceinline__ int unit_of(int f) { return f >> 3; }
    static __device__ __forceinline__ int quad_of(int f) { return f & 7; }
    static __device__ __forceinline__ void load_acts(X &x, const float4 *p, int stride) { load_x(p, stride, x.v, 32); }
    static __device__ __forceinline__ void load(Regs &w, const DevTensor &W, size_t u0, uint32_t i) {
        const uint8_t *q = W.p0 + u0 * 32;
        w.q0 = ldg16(q + i * 32u);
        w.q1 = ldg16(q + i * 32u + 16u);
        w.d = *reinterpret_cast<const uint16_t *>(W.p1 + u0 * 2 + i * 2u);
    }
    static __device__ __forceinline__ float dot(const Regs &w, int, const X &x) {
        const uint32_t q[8] = {w.q0.x, w.q0.y, w.q0.z, w.q0.w, w.q1.x, w.q1.y, w.q1.z, w.q1.w};
        float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 8; t++) {
            s[0] = fmaf((float)(int8_t)(q[t] & 0xffu), x.v[4 * t], s[0]);
            s[1] = fmaf((float)(int8_t)((q[t] >> 8) & 0xffu), x.v[4 * t + 1], s[1]);
            s[2] = fmaf((float)(int8_t)((q[t] >> 16) & 0xffu), x.v[4 * t + 2], s[2]);
            s[3] = fmaf((float)(int8_t)(q[t] >> 24), x.v[4 * t + 3], s[3]);
        }
        return f16_bits_to_f32(w.d) * ((s[0] + s[1]) + (s[2] + s[3]));
    }
};

struct FmtQ4_K {
    static constexpr int kElems = 64, ND = 2;
    static constexpr double kRound = 0.9, kLanes = 1024, kKeep = 0.94, kLong = 6;
    static int waves(int) { return 16; }
    static bool takes(int, int nd, bool runs) { return nd == 1 || runs; }
    struct X {
        float v[64], s[4];  // the activations and the sums of their groups of 16
    };
    struct Regs {
        uint4 q0, q1;
        uint32_t h;  // header word u % 4; the four units of a super-block share theirs over DPP
    };
    static __device__ __forceinline__ int unit_of(int f) { return f >> 4; }
    static __device__ __forceinline__ int quad_of(int f) { return f & 15; }
    static __device__ __forceinline__ void load_acts(X &x, const float4 *p, int stride) {
        load_x(p, stride, x.v, 64);
#pragma unroll
        for (int q = 0; q < 4; q++) x.s[q] = sum16(x.v + 16 * q);
    }
    static __device__ __forceinline__ void load(Regs &w, const DevTensor &W, size_t u0, uint32_t i) {
        const uint8_t *q = W.p1 + u0 * 32;
        w.q0 = ldg16(q + i * 32u);
        w.q1 = ldg16(q + i * 32u + 16u);
        w.h = *reinterpret_cast<const uint32_t *>(W.p0 + u0 * 4 + i * 4u);
    }
    static __device__ __forceinline__ float dot(const Regs &w, int p, const X &x) {
        uint32_t h0, h1, h2, h3;
        quad_header(w.h, h0, h1, h2, h3);
        const PairScale s = pair_scale(h0, h1, h2, h3, p);
        const uint32_t q[8] = {w.q0.x, w.q0.y, w.q0.z, w.q0.w, w.q1.x, w.q1.y, w.q1.z, w.q1.w};
        // two chains per group of 16, low nibbles (l) and high ones (u, as 16 q)
        float l[4] = {0.f, 0.f, 0.f, 0.f}, u[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const uint32_t q8 = q[t] >> 8;
            const int c = 2 * (t >> 2);
            l[c] = fma_codes(q[t] & 0x000f000fu, x.v[4 * t], x.v[4 * t + 2], l[c]);
            l[c + 1] = fma_codes(q8 & 0x000f000fu, x.v[4 * t + 1], x.v[4 * t + 3], l[c + 1]);
            u[c] = fma_codes(q[t] & 0x00f000f0u, x.v[32 + 4 * t], x.v[32 + 4 * t + 2], u[c]);
            u[c + 1] = fma_codes(q8 & 0x00f000f0u, x.v[32 + 4 * t + 1], x.v[32 + 4 * t + 3], u[c + 1]);
        }
        const float s0 = s.dsc0 * 0x1p24f, s1 = s.dsc1 * 0x1p20f;
        return ((s0 * (l[0] + l[1]) - s.dmn0 * x.s[0]) + (s0 * (l[2] + l[3]) - s.dmn0 * x.s[1])) +
               ((s1 * (u[0] + u[1]) - s.dmn1 * x.s[2]) + (s1 * (u[2] + u[3]) - s.dmn1 * x.s[3]));
    }
};

struct FmtQ6_K {
    static constexpr int kElems = 64, ND = 2;
    static constexpr double kRound = 1.0, kLanes = 1024, kKeep = 0.94, kLong = 6;
    static int waves(int) { return 16; }
    static bool takes(int, int nd, bool runs) { return nd == 1 || runs; }
    struct X {
        float v[64], s[4];  // four groups of 16, and -32 times their sums
    };
    struct Regs {
        uint4 qa, qb, qh;
        uint2 sc;
        uint16_t d;
    };
    // unit 4 sb + 2 hf + l holds elements 256 sb + 128 hf + 16 l + 32 q + [0, 16), q < 4
    static __device__ __forceinline__ int unit_of(int f) { return (f >> 5) * 2 + ((f >> 2) & 1); }
    static __device__ __forceinline__ int quad_of(int f) { return ((f >> 3) & 3) * 4 + (f & 3); }
    static __device__ __forceinline__ void load_acts(X &x, const float4 *p, int stride) {
        load_x(p, stride, x.v, 64);
#pragma unroll
        for (int q = 0; q < 4; q++) x.s[q] = -32.0f * sum16(x.v + 16 * q);
    }
    static __device__ __forceinline__ void load(Regs &w, const DevTensor &W, size_t u0, uint32_t i) {
        const size_t b0 = u0 >> 2;
        const uint32_t b = i >> 2, hf = (i >> 1) & 1u, l0 = (i & 1u) * 16u;
        w.qa = ldg16_nt(W.p0 + b0 * 128 + (b * 128u + 64u * hf + l0));
        w.qb = ldg16_nt(W.p0 + b0 * 128 + (b * 128u + 64u * hf + 32u + l0));
        w.qh = ldg16_nt(W.p1 + b0 * 64 + (b * 64u + 32u * hf + l0));
        w.sc = *reinterpret_cast<const uint2 *>(W.p2 + b0 * 16 + (b * 16u + 8u * hf));
        w.d = *reinterpret_cast<const uint16_t *>(W.p3 + b0 * 2 + b * 2u);
    }
    static __device__ __forceinline__ float dot(const Regs &w, int p, const X &x) {
        const uint32_t sa[4] = {w.qa.x, w.qa.y, w.qa.z, w.qa.w};
        const uint32_t sb[4] = {w.qb.x, w.qb.y, w.qb.z, w.qb.w};
        const uint32_t sh[4] = {w.qh.x, w.qh.y, w.qh.z, w.qh.w};
        const int is = p & 1;
        const float d = f16_bits_to_f32(w.d);
        float acc = 0.f;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            float s0 = 0.f, s1 = 0.f;
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const uint32_t lo = q == 0   ? sa[t] & 0x0f0f0f0fu
                                    : q == 1 ? sb[t] & 0x0f0f0f0fu
                                    : q == 2 ? (sa[t] >> 4) & 0x0f0f0f0fu
                                             : (sb[t] >> 4) & 0x0f0f0f0fu;
                const uint32_t hi = q == 0 ? sh[t] << 4 : q == 1 ? sh[t] << 2 : q == 2 ? sh[t] : sh[t] >> 2;
                const uint32_t g = lo | (hi & 0x30303030u);
                const float *v = x.v + 16 * q + 4 * t;
                s0 = fma_codes(g & 0x003f003fu, v[0], v[2], s0);
                s1 = fma_codes((g >> 8) & 0x003f003fu, v[1], v[3], s1);
            }
            const int bi = is + 2 * q;  // byte of the half's 8 scale bytes
            const float scale = (float)(int8_t)(((bi < 4 ? w.sc.x : w.sc.y) >> (8 * (bi & 3))) & 0xffu);
            acc = fmaf(d * scale, fmaf(0x1p24f, s0 + s1, x.s[q]), acc);
        }
        return acc;
    }
};

}  // namespace lt
