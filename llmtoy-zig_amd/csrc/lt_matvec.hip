// lt_matvec.hip -- matvec over rows of any length with fp32 activations:
// Q8_0, and Q4_K / Q6_K rows that the streaming kernels (lt_q4k.hip,
// lt_q6k.hip: 1, 2, 4, 8 or 16 super-blocks) do not take.
//
// A row is U work units (Q8_0: a 32-element block; K-quants: 64 elements, a
// Q4_K sub-block pair or a quarter of a Q6_K super-block).  A thread keeps
// one unit position for the whole launch, so its activations stay in
// registers; a workgroup of as many wavefronts as waste the fewest lanes
// takes RP = threads / U whole rows side by side (a pass) and walks the
// matrix with ND passes in flight.  A row's lanes may straddle wavefronts:
// the partial sums of ND passes meet in LDS after one barrier.
//
// What bounds it: HBM on large matrices, the launch and a round trip to
// memory on small ones.  Measured (us a launch, cold weights, the kernels
// this replaces -> here): Q6_K 262,144 x 2,816 188 -> 115 (5.3 TB/s), 4,096 x
// 2,816 7.9 -> 5.8; Q4_K 40,000 x 2,560 23.1 -> 17.7, 4,096 x 2,816 7.5 ->
// 5.2, 2,048 x 5,120 10.4 -> 5.5; Q8_0 7,001 x 2,816 9.3 -> 7.6, 4,096 x
// 4,096 10.2 -> 6.4, 151,936 x 896 31.0 -> 26.8, 600 x 512 2.3 -> 2.4.  The
// old kernels put a power of two of lanes on a row (11 super-blocks: a third
// of them idle), waited for x before they requested a weight, and converted
// every code.  Activations as three int8 limbs against v_dot4 instead were
// slower (Q6_K 142 us: the conversion and 14 LDS reads a unit) and less
// exact (2.5e-7 from 64 bits, 1.9e-7 before, 1.6e-7 here).
#include "lt_internal.h"
#include "lt_limbs.h"

#include <algorithm>

namespace lt {

namespace {

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
// of unit i behind unit u0 of the matrix, and the unit's dot product.
struct FmtQ8_0 {
    static constexpr int kElems = 32, ND = 4;
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

// A pass is RP rows of U units on nthreads = blockDim threads; T = 2^logT
// threads add up a row.
struct RowsPlan {
    int U, RP, nthreads, nblk, logT, npass;
};

}  // namespace

// Pass ps covers rows RP ps + [0, RP); workgroup b takes passes b, b +
// gridDim.x, ... in rounds of ND (one load buffer each).  Thread t < RP U
// works on row t / U of a pass at unit t % U.  The activations come through
// LDS, quad by quad ([quad][unit]: a wavefront's reads have no bank
// conflicts), requested ahead of the first weights so that the wait for them
// does not include those.  Loads are unconditional (clamped to the last
// row), but the last round loads nothing.  IN_WAVE: U is a power of two up
// to 64, a row's lanes are neighbours in one wavefront; else the partial
// sums of a round meet in part, which is double-buffered: a round's sums are
// read behind its barrier, and the buffer is written again two rounds later.
template <class F, int ND, bool IN_WAVE>
__global__ void __launch_bounds__(512, 4) k_matvec_rows(DevTensor W, const float *__restrict__ x,
                                                        float *__restrict__ y, RowsPlan p) {
    __shared__ float part[IN_WAVE ? 1 : 2][IN_WAVE ? 1 : ND][IN_WAVE ? 1 : 512];
    extern __shared__ float4 xs[];
    const int tid = threadIdx.x, NT = p.nthreads, U = p.U;
    const int r = min(tid / U, p.RP - 1), u = tid % U;
    const int nrows = (int)W.total_rows;
    typename F::Regs w[ND];
    auto ld = [&](typename F::Regs &rg, int ps) {
        const int row0 = min(ps * p.RP, nrows - 1);  // (uniform)
        F::load(rg, W, (size_t)row0 * U, (uint32_t)(min(r, nrows - 1 - row0) * U + u));
    };
    const int stride = gridDim.x;
    int ps = blockIdx.x;
    const int nf = (int)W.cols / 4, fa = min(tid, nf - 1), fb = min(tid + NT, nf - 1);
    const float4 f0 = ldg16f(x + 4 * fa), f1 = ldg16f(x + 4 * fb);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < ND; i++) ld(w[i], ps + i * stride);
    __builtin_amdgcn_sched_barrier(0);
    xs[F::quad_of(fa) * U + F::unit_of(fa)] = f0;
    xs[F::quad_of(fb) * U + F::unit_of(fb)] = f1;
    for (int f = tid + 2 * NT; f < nf; f += NT) xs[F::quad_of(f) * U + F::unit_of(f)] = ldg16f(x + 4 * f);
    __syncthreads();
    typename F::X xv;
    F::load_acts(xv, xs + u, U);
    const int T = 1 << p.logT, rpr = ND * p.RP;  // threads a row and rows of a round's sums
    int buf = 0;
    auto round = [&](bool more) {
#pragma unroll
        for (int i = 0; i < ND; i++) {
            float t = F::dot(w[i], u & 3, xv);
            if (more) ld(w[i], ps + (ND + i) * stride);
            if (IN_WAVE) {
                for (int off = T >> 1; off > 0; off >>= 1) t += __shfl_xor(t, off, kWave);
                const int out = (ps + i * stride) * p.RP + r;
                if (u == 0 && out < nrows) y[out] = t;
            } else {
                part[buf][i][tid] = t;
            }
        }
        if (!IN_WAVE) {
            __syncthreads();
            for (int q = tid >> p.logT; q < rpr; q += NT >> p.logT) {
                const int i = q / p.RP, rr = q - i * p.RP, o = tid & (T - 1);
                float sum = 0.f;
                for (int v = o; v < U; v += T) sum += part[buf][i][rr * U + v];
                for (int off = T >> 1; off > 0; off >>= 1) sum += __shfl_xor(sum, off, kWave);
                const int out = (ps + i * stride) * p.RP + rr;
                if (o == 0 && out < nrows) y[out] = sum;
            }
            buf ^= 1;
        }
        ps += ND * stride;
    };
    while (ps + ND * stride < p.npass) round(true);
    round(false);
}

namespace {

template <class F, int ND, bool IN_WAVE>
hipError_t launch_rows_t(const DevTensor &W, const float *x, float *y, RowsPlan &p, hipStream_t s) {
    p.logT = 0;
    if (IN_WAVE)
        while ((1 << p.logT) < p.U) p.logT++;
    else
        while (p.logT < 6 && (2 << p.logT) <= p.U && (ND * p.RP << (p.logT + 1)) <= p.nthreads) p.logT++;
    hipLaunchKernelGGL((k_matvec_rows<F, ND, IN_WAVE>), dim3(p.nblk), dim3(p.nthreads), W.cols * 4, s, W, x, y, p);
    return hipGetLastError();
}

template <class F>
hipError_t launch_rows(const DevTensor &W, const float *x, float *y, hipStream_t s) {
    RowsPlan p{};
    p.U = (int)W.cols / F::kElems;
    if (p.U > 512 || W.total_rows >= (size_t)1 << 30) return hipErrorInvalidValue;
    // The workgroup size that leaves the fewest lanes idle, the largest of
    // them: x is staged once per workgroup (Q4_K 4,096 x 11,008 on 512 threads
    // 11.6 us, on 256 14.9; Q8_0 7,001 x 2,816 7.6 and 8.2).  A short matrix
    // takes smaller ones until about 96 have a pass each (Q4_K 1,000 x 1,536:
    // 3.9 us on 512, 3.4 on 256).
    double best = 0;
    for (int nt = 512; nt >= 128 && nt >= p.U; nt -= 64) {
        const int rp = nt / p.U, npass = (int)((W.total_rows + rp - 1) / rp);
        const double used = (double)(rp * p.U) / nt * (npass >= 96 ? 1.0 : npass / 96.0);
        if (used > best * 1.01) {
            best = used;
            p.nthreads = nt;
        }
    }
    p.RP = p.nthreads / p.U;
    p.npass = (int)((W.total_rows + p.RP - 1) / p.RP);
    const int cap = 256 * (1024 / p.nthreads);  // resident workgroups: 16 wavefronts a CU
    p.nblk = std::min(p.npass, cap);
    // up to two passes a workgroup: one load buffer, as the others would load
    // rows again that nobody needs (Q8_0 4,096 x 4,096: 6.3 us, 7.1 with four)
    const bool one = p.npass <= 2 * cap;
    if (p.U <= 64 && (p.U & (p.U - 1)) == 0)
        return one ? launch_rows_t<F, 1, true>(W, x, y, p, s) : launch_rows_t<F, F::ND, true>(W, x, y, p, s);
    return one ? launch_rows_t<F, 1, false>(W, x, y, p, s) : launch_rows_t<F, F::ND, false>(W, x, y, p, s);
}

}  // namespace

hipError_t launch_matvec_rows(const DevTensor &W, const float *x, float *y, hipStream_t s) {
    switch (W.type) {
    case 8: return launch_rows<FmtQ8_0>(W, x, y, s);
    case 12: return launch_rows<FmtQ4_K>(W, x, y, s);
    case 14: return launch_rows<FmtQ6_K>(W, x, y, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace lt
