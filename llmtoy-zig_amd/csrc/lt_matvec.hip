// lt_matvec.hip -- matvec over rows of any length with fp32 activations:
// Q8_0, and the Q4_K / Q6_K matrices that the streaming kernels (lt_q4k.hip,
// lt_q6k.hip: rows of 1, 2, 4, 8 or 16 super-blocks, and enough of them) do
// not take.
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
// 2,816 6.9 -> 5.5; Q4_K 40,000 x 2,560 21.0 -> 16.7, 4,096 x 2,816 6.6 ->
// 4.9, 2,816 x 5,120 9.1 -> 5.9; Q8_0 7,001 x 2,816 8.0 -> 6.9, 4,096 x
// 4,096 9.0 -> 6.0, 152,000 x 2,048 62 -> 62, 152,000 x 896 33 -> 27.  The
// old kernels put a power of two of lanes on a row (11 super-blocks: a third
// of them idle), waited for x before they requested a weight, and converted
// every code.  Activations as three int8 limbs against v_dot4 instead were
// slower (Q6_K 142 us: the conversion and 14 LDS reads a unit) and less
// exact (2.5e-7 from 64 bits, 1.9e-7 before, 1.6e-7 here).
#include "lt_rows.h"

#include <algorithm>

namespace lt {

namespace {

// A pass is RP rows of U units on nthreads = blockDim threads; T = 2^logT
// threads add up a row; nd load buffers.
struct RowsPlan {
    int U, RP, nthreads, nblk, logT, npass, nd;
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

// A launch of nt threads a workgroup and nd load buffers, on up to waves
// wavefronts a CU.
RowsPlan rows_plan(int rows, int U, int nt, int nd, int waves) {
    RowsPlan p{};
    p.U = U;
    p.nthreads = nt;
    p.RP = nt / U;
    p.npass = (rows - 1) / p.RP + 1;
    p.nblk = std::min(p.npass, 256 * (waves * 64 / nt));
    p.nd = nd;
    return p;
}

// An estimate of the launch, as bytes that the CU with the most passes reads:
// its weights, with passes in rounds of nd (F::kRound of the time, as more is
// in flight), times (F::kLanes / lanes)^3 where the matrix fills the chip and
// the lanes at work on a CU are fewer than that; twice the x that its
// workgroups stage; and 3,000 for every round of x loads behind the two quads
// a thread that go ahead of the weights.  Fitted to 570 sizes: the shape of
// the least estimate takes 1.03 of the best shape's time on the average.
template <class F>
double rows_cost(const RowsPlan &p, int cols, double row_bytes) {
    // workgroups of that CU, as LDS (160 KB) lets them be resident
    const int per_cu = std::min((p.nblk + 255) / 256, (160 << 10) / (cols * 4 + p.nd * 4096));
    auto whole = [&](int n) { return (n + p.nd - 1) & ~(p.nd - 1); };  // passes in whole rounds
    int passes = per_cu * p.nd;
    double few = 1.0;
    if (p.npass > 256 * per_cu) {
        const int n = p.npass / (256 * per_cu), more = (p.npass - n * 256 * per_cu + 255) / 256;
        passes = more * whole(n + 1) + (per_cu - more) * whole(n);
        few = std::max(1.0, F::kLanes / (per_cu * p.RP * p.U));
    }
    const int late = std::max(0, (cols / 4 - p.nthreads - 1) / p.nthreads);
    return passes * (p.RP * row_bytes) * (p.nd > 1 ? F::kRound : 1.0) * (few * few * few) + 8.0 * per_cu * cols +
           3000.0 * late;
}

template <class F>
hipError_t launch_rows(const DevTensor &W, const float *x, float *y, hipStream_t s) {
    const int cols = (int)W.cols, rows = (int)W.total_rows, U = cols / F::kElems;
    // row indices are ints, and a last round's go up to 2 ND cap passes (2^21 rows) past the end
    if (U > 512 || W.total_rows > ((size_t)1 << 31) - (1 << 22)) return hipErrorInvalidValue;
    // up to two passes a workgroup: one load buffer, as the others would load
    // rows again that nobody needs (Q8_0 4,096 x 4,096: 6.3 us, 7.1 with four)
    auto runs = [&](int npass, int nt) { return npass > 2 * 256 * (1024 / nt); };
    // The workgroup size that leaves the fewest lanes idle, the largest of
    // them: x is staged once per workgroup (Q4_K 4,096 x 11,008 on 512 threads
    // 11.6 us, on 256 14.9; Q8_0 7,001 x 2,816 7.6 and 8.2).  A short matrix
    // takes smaller ones until 160 have a pass each (Q6_K 4,096 x 512: 3.19 us,
    // 3.84 with 96, 3.11 with 256; 6,000 x 512 3.30, 4.02, 3.56), but less
    // willingly where x is more than the two quads a thread that go ahead of
    // the weights (Q6_K 1,000 x 1,536: 3.37 us on 192 threads, 3.71 on 128; Q8_0
    // 200 x 4,096: 3.36 on 256, 3.70 on 128).
    double best = 0;
    RowsPlan p{};
    for (int nt = 512; nt >= 128 && nt >= U; nt -= 64) {
        RowsPlan q = rows_plan(rows, U, nt, 1, 16);
        if (runs(q.npass, nt)) q.nd = F::ND;
        const double used = (double)(q.RP * U) / nt * (q.npass >= 160 ? 1.0 : q.npass / 160.0) *
                            (cols <= 8 * nt ? 1.0 : cols <= 16 * nt ? 0.75 : 0.4);
        if (used > best * 1.01) {
            best = used;
            p = q;
        }
    }
    // That shape does not see passes that go unevenly over the CUs, or come in
    // whole rounds: another one whose estimate is clearly less (F::kKeep) takes
    // its place, but for K-quants not in long runs, where unevenness is small and
    // the estimate errs by as much (Q6_K 262,144 x 2,816: 114 us kept, 131
    // replaced).  Kept | replaced, us: Q6_K 7,001 x 5,120 15.9 | 10.1; Q4_K 16,000 x
    // 1,280 7.2 | 5.7, 7,001 x 5,120 12.4 | 8.6; Q8_0 152,000 x 512 19.4 | 16.1,
    // 11,000 x 2,048 8.5 | 6.8, 2,816 x 4,864 7.2 | 6.4; the other way Q4_K 16,000 x
    // 1,792 6.6 | 7.1, Q6_K 11,000 x 1,536 6.3 | 6.6.
    if (p.npass <= F::kLong * p.nblk) {
        const double row_bytes = (double)W.bytes / rows;
        double least = F::kKeep * rows_cost<F>(rows_plan(rows, U, p.nthreads, p.nd, p.nd == 1 ? F::waves(U) : 16), cols,
                                               row_bytes);
        for (int nt = 512; nt >= 128 && nt >= U; nt -= 64)
            for (int nd : {1, F::ND}) {
                const RowsPlan q = rows_plan(rows, U, nt, nd, nd == 1 ? F::waves(U) : 16);
                if (!F::takes(U, nd, runs(q.npass, nt))) continue;
                const double cost = rows_cost<F>(q, cols, row_bytes);
                if (cost < least) {
                    least = cost;
                    p = q;
                }
            }
    }
    if (U <= 64 && (U & (U - 1)) == 0)
        return p.nd == 1 ? launch_rows_t<F, 1, true>(W, x, y, p, s) : launch_rows_t<F, F::ND, true>(W, x, y, p, s);
    return p.nd == 1 ? launch_rows_t<F, 1, false>(W, x, y, p, s) : launch_rows_t<F, F::ND, false>(W, x, y, p, s);
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
