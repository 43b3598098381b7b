// lt_prefill.hip -- batched prefill of one MoE layer (Q4_K experts) on MFMA.
//
// The reference prefills one token at a time through the decode path
// (main.zig:1916-1922).  Here T tokens go through the layer together:
//   1. router logits for all tokens with the reference's exact dotf32 order
//      and per-token softmax / top-k (lt_router.hip);
//   2. dispatch: a block per expert lays its rows out behind those of the
//      experts before it ("sorted rows"), cuts them into chunks of at most
//      MC = 64, and places its (token, slot) assignments in assignment order
//      (a stable counting sort);
//      X is converted to f16 once (by the router kernel, or
//      k_prefill_x_f16), each row t divided by r_t = 2^e, a power of two
//      that puts its largest element in [1, 2);
//   3. grouped gate/up GEMM: one block per (chunk, 64 output columns), a
//      wavefront of it per 16 columns: its 32 weight rows (16 gate + the
//      matching 16 up) are dequantised from Q4_K to f16 in registers, as the
//      B operand of v_mfma_f32_32x32x16_f16 (fp32 accumulation), and meet the
//      chunk's one or two 32-row token tiles, which the block shares through
//      LDS.  Gate and up of an output column sit in the same wavefront, so
//      the epilogue h = act(gate) * up exchanges values between two halves
//      of a row only; it stores H = h / r_t^2 (f16), which |act(g)| <= |g|
//      bounds by the scaled row's products whatever X's magnitude (a value
//      still past f16's range saturates at +-65504 and is counted: the call
//      then reports LT_ERR_DEVICE);
//   4. grouped down GEMM: one block per (chunk, 128 output rows), the same
//      scheme with H as the token operand -> Y (fp32, sorted rows);
//   5. combine: out[t] = r_t^2 * sum over slots in slot order of w[t][s] *
//      Y[pos] (r_t^2 exact).
// Steps 3 and 4 run as one launch when blocks with equal index % 8 share an
// XCD (k_prefill_gemms: a chunk's down blocks take H from its gate/up
// blocks through that XCD's L2), else as two.  Chunks of a single token
// skip the tiles: their blocks stream the weights against int8 limbs of the
// token like the decode kernels (gate_up_tiny, down_tiny).
// Both GEMMs run over K stages of 64 (a pair of Q4_K sub-blocks): weights
// are requested a super-block ahead, tokens two stages ahead into registers
// and one into a double buffer in LDS, and each stage ends in one barrier.
// The fp32 sums of a row run in K order whatever its chunk; only the
// one-token stream sums in another order, and the stable placement gives
// every row the same chunk on every call, so the output is bit-identical run
// to run.
//
// Why this shape (Q4_K experts of 2048 x 768, 128 of them, 8 a token, both
// GEMMs in one launch): the work is bound by the vector instructions that
// dequantise, the clock falls under the load, and a batch of 512 tokens
// leaves 32 rows an expert.  Eight wavefronts that dequantised 128 rows
// into f16 LDS tiles for chunks of 128 rows spent most of their time at the
// barrier behind the dequantisation and filled half a tile: 512 tokens took
// 166 us, 1024 251 us, 37 79.6 us (whole calls); 64-row chunks, a fragment
// dequantised where it is used and four small blocks a CU that cover each
// other's waits: 143 us, 219 us, 71 us.  Wavefronts that held 128 rows each
// (two blocks a CU, half the dequantisation for full chunks) measured 156 us
// and 226 us: the batch rarely fills them.  Long batches, where experts do
// fill 128 rows, are faster too, with even routing as with a skewed one: 2,048
// tokens 422 -> 360 us, 4,096 743 -> 650, 16,384 2,910 -> 2,440.
//
// f16 rather than bf16 tiles: a Q4_K nibble q becomes the exact f16 1024 + q
// (or 1024 + 16 q) with one v_and_or (its bits in the mantissa under 1024's
// exponent), two such values per dword, so the dequantisation is a packed
// f16 subtract of 1024 and a packed f16 fma (d sc) q - dmin mn per pair of
// weights, with no conversion or packing step -- and f16 keeps 3 more
// mantissa bits than bf16.  The pairs come out as elements (0, 2) and (1, 3) of each aligned
// group of 4, so every K dimension is stored with the middle two of each 4
// swapped (kperm): X and H are written in that order, and the MFMA sums the
// same products.
#include "lt_internal.h"
#include "lt_limbs.h"

#include <stdlib.h>

namespace lt {

typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

namespace {

constexpr int MC = 64;        // sorted rows per chunk: one or two token tiles of 32
constexpr int KS = 64;        // K per stage: a sub-block pair of a Q4_K super-block
constexpr int PT = 256;       // threads of a GEMM block: 4 wavefronts of 32 weight rows
constexpr int BN1 = 64;       // gate/up output columns per block (16 a wavefront)
constexpr int BN2 = 128;      // down output rows (= output columns of Y) per block

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

struct Ws {
    float *logits;
    uint32_t *ids;
    float *w;
    int *chunks;    // [max_chunks][3] = (expert, first sorted row, rows)
    int *n_chunks;  // [1]
    int *perm;      // [T*k] token of each sorted row
    int *pos;       // [T*k] sorted row of assignment t*k + s
    float *rs;      // [T] row scales: X row t = rs[t] * Xh row t
    _Float16 *Xh;   // [T][D] X / rs in f16, columns in kperm order
    _Float16 *H;    // [T*k][Kd], columns in kperm order
    float *Y;       // [T*k][D]
    int *done;      // [max_chunks] finished gate/up blocks per chunk (fused GEMMs)
};

int max_chunks(int TK, int E) { return (TK + MC - 1) / MC + E; }

Ws carve(void *base, int T, int k, int E, int Kd, int D) {
    uint8_t *p = (uint8_t *)base;
    const size_t TK = (size_t)T * k;
    Ws w;
    w.logits = (float *)p; p += align256((size_t)T * E * 4);
    w.ids = (uint32_t *)p; p += align256(TK * 4);
    w.w = (float *)p; p += align256(TK * 4);
    w.chunks = (int *)p; p += align256((size_t)max_chunks((int)TK, E) * 12);
    w.n_chunks = (int *)p; p += 256;
    w.perm = (int *)p; p += align256(TK * 4);
    w.pos = (int *)p; p += align256(TK * 4);
    w.rs = (float *)p; p += align256((size_t)T * 4);
    w.Xh = (_Float16 *)p; p += align256((size_t)T * D * 2);
    w.H = (_Float16 *)p; p += align256(TK * Kd * 2);
    w.Y = (float *)p; p += align256(TK * D * 4);
    w.done = (int *)p; p += align256((size_t)max_chunks((int)TK, E) * 4);
    return w;
}

// LDS token tiles: a row's 64 K values are 8 units of 8 f16 (16 bytes); unit u
// of row r is stored at unit u ^ aswz(r), so that the MFMA operand reads
// (consecutive lanes: consecutive rows, one unit) of 16 rows fall in distinct
// 16-byte bank groups (two rows to the 64 banks).
__host__ __device__ __forceinline__ int aswz(int r) { return (r >> 1) & 7; }

// The K order of every f16 operand: within each aligned group of 4 the
// middle two elements are swapped (an involution).
__host__ __device__ __forceinline__ int kperm(int c) { return (c & ~3) | ((c & 1) << 1) | ((c >> 1) & 1); }

// The (1024 + q 2^j) pairs of a fragment -> (scale q + neg_min) pairs (scale
// already divided by 2^j): 8 weights of the MFMA's B operand.
__device__ __forceinline__ f16x8 q4_frag(uint32_t v0, uint32_t v1, uint32_t v2, uint32_t v3, half2v sc, half2v nm) {
    const half2v k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
    const uint32_t v[4] = {v0, v1, v2, v3};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const half2v q = __builtin_bit_cast(half2v, v[i]) - k1024;  // exact: q 2^j, q in 0..15
        o[i] = __builtin_bit_cast(uint32_t, q * sc + nm);
    }
    return __builtin_bit_cast(f16x8, make_uint4(o[0], o[1], o[2], o[3]));
}

struct NoWait {
    __device__ __forceinline__ void operator()() const {}
};

// LDS of a GEMM block (40 KB: four blocks a CU): the token tiles' two stages
// (after the GEMM the chunk's row scales), and per wavefront one super-block
// of its 32 weight rows as loaded (128 bytes a row) and the headers of up to
// 4 super-blocks (16 bytes each, 64 a row).
struct __attribute__((aligned(16))) GemmLds {
    _Float16 tok[2 * MC * KS];
    uint4 quants[PT / 64][256], heads[PT / 64][128];
};

// The grouped GEMM of one wavefront: its 32 weight rows against the chunk's
// MT token tiles of 32, K = 256 nsb.  Every wavefront of the block works on
// the same tokens and rows of its own.
// Weights: the MFMA wants lane l to hold row l & 31, whose rows are a row
// length apart in memory -- loaded that way each 16-byte load touches 32
// cache lines and takes about 100 cycles of the CU's load path, more than the
// MFMAs that use it.
// So eight lanes load a row's 128 bytes, eight rows a load, and the words
// cross to their lanes through a buffer in LDS that only this wavefront uses;
// the LDS sees a wavefront's accesses in order, so a super-block is written
// as soon as the one before has been read.  goff[j] is the byte offset of row
// 8 j + (lane >> 3) in the quant plane (8 times that in the header plane).
// Dequantised (quant/dequant.zig:157-187: (d*sc)*q - dmin*mn) straight into
// the B fragments, the weights are never written again.  K is taken in the
// order the nibbles come: the lane's 16 bytes of pair p are bytes 16 (lane >>
// 5) of the pair's 32, and fragment (pair, low or high nibble, half j of the
// 16) holds elements 64 p + 32 hi + 16 (lane >> 5) + 8 j + [0, 8), each
// aligned 4 with its middle two swapped (kperm); the token tile is read in
// the same order.  Under f16's exponent of 1024 (0x6400) a nibble in mantissa
// bits 0-3 reads 1024 + q and one in bits 4-7 reads 1024 + 16 q, both exact:
// one v_and_or a pair of weights (the masks kept in registers so that the
// compiler forms it), the high nibbles' scale divided by 16.
// Tokens: each thread loads 16 bytes of one row of every tile a stage (K =
// 64) into registers, two stages ahead, and writes them to the LDS buffer
// that the stage before has read; one barrier a stage.  aoff counts units of
// 16 bytes (65536 rows of any length pass 4 GB).
// All loads are unconditional (stages past the end clamped, their data left
// unused), so that the waits count what is in flight.  wait() runs in every
// thread once the first weights are requested and before the first token
// load.
template <int MT, typename Wait>
__device__ __forceinline__ void gemm_tiles(floatx16 (&acc)[MT], GemmLds &L, const uint8_t *hdr, const uint8_t *qs,
                                           uint32_t up, int nsb, const uint8_t *abase, const uint32_t (&aoff)[MT],
                                           int wave, int tid, int lane, Wait wait) {
    constexpr int TB = MT * 32 * KS;  // f16 per token buffer
    constexpr bool kWaits = !__is_same(Wait, NoWait);
    const int NS = 4 * nsb;
    uint4 Q[4], A[2][MT];
    const int lr = lane >> 3, lc = lane & 7;  // a load's row 8 j + lr, word lc
    const int row = lane & 31, half = lane >> 5;
    // rows 8 j + lr of the wavefront's weights: j = 2, 3 are `up` rows behind j = 0, 1
    const uint32_t pitch = (uint32_t)nsb * 128u, goff = (uint32_t)lr * pitch + 16u * lc;
    auto jrow = [&](int j) { return (j & 1) * 8u + (j >= 2 ? up : 0u); };
    auto qld = [&](int sb) {
        const uint8_t *p = qs + (size_t)min(sb, nsb - 1) * 128;
#pragma unroll
        for (int j = 0; j < 4; j++) Q[j] = ldg16(p + (size_t)jrow(j) * pitch + goff);
    };
    // word c of row r stands at byte 128 r + 16 (c ^ (r >> 1 & 7)) of the
    // wavefront's quants: for row 8 j + lr that is 1024 j + 128 lr + 16 ((lc ^
    // lr >> 1) ^ 4 (j & 1)), so that one address register serves all four
    uint8_t *const wq = reinterpret_cast<uint8_t *>(L.quants[wave]);
    const uint32_t qwr = 128u * lr + 16u * (lc ^ (lr >> 1)), qrd = 128u * row + 16u * (half ^ ((row >> 1) & 7));
    auto qput = [&] {
        const uint32_t b = opaque(qwr);
#pragma unroll
        for (int j = 0; j < 4; j++) *reinterpret_cast<uint4 *>(wq + ((b ^ (64u * (j & 1))) + 1024u * j)) = Q[j];
    };
    // headers of super-blocks sb + [0, 4), word c of row r at byte 64 r + 16
    // (c ^ (r >> 2 & 3)): lane words 0-3 load rows 8 j + lr for j = 0, 1, the
    // others for j = 2, 3
    uint8_t *const wh = reinterpret_cast<uint8_t *>(L.heads[wave]);
    const int hr = 16 * (lc >> 2) + lr, hc = lc & 3;
    auto hld = [&](uint4 (&r)[2], int sb) {
        const uint8_t *p =
            hdr + (size_t)min(sb + hc, nsb - 1) * 16 + (size_t)((lc >> 2 ? up : 0u) + lr) * (uint32_t)(nsb * 16);
        r[0] = ldg16(p);
        r[1] = ldg16(p + nsb * 128);
    };
    auto hput = [&](const uint4 (&r)[2]) {
        *reinterpret_cast<uint4 *>(wh + 64 * hr + 16 * (hc ^ ((hr >> 2) & 3))) = r[0];
        *reinterpret_cast<uint4 *>(wh + 64 * (hr + 8) + 16 * (hc ^ (((hr + 8) >> 2) & 3))) = r[1];
    };
    const uint32_t hrd = 64u * row + 16u * ((row >> 2) & 3);
    auto ald = [&](uint4 (&r)[MT], int st) {
        const uint32_t k = (uint32_t)min(st, NS - 1) * (KS / 8);
#pragma unroll
        for (int t = 0; t < MT; t++) r[t] = ldg16(abase + ((uint64_t)(aoff[t] + k) << 4));
    };
    _Float16 *const aw = L.tok + (tid >> 3) * KS + 8 * ((tid & 7) ^ aswz(tid >> 3));
    auto awr = [&](const uint4 (&r)[MT], int buf) {
#pragma unroll
        for (int t = 0; t < MT; t++) *reinterpret_cast<uint4 *>(aw + buf * TB + t * 32 * KS) = r[t];
    };
#pragma unroll
    for (int t = 0; t < MT; t++) acc[t] = floatx16{};
    uint4 h0[2];
    hld(h0, 0);
    qld(0);
    if (!kWaits) {
        ald(A[0], 0);
        ald(A[1], 1);
    }
    hput(h0);
    qput();
    qld(1);
    if (kWaits) {
        wait();
        ald(A[0], 0);
        ald(A[1], 1);
    }
    awr(A[0], 0);
    ald(A[0], 2);
    // fragment (pp, hi, j) of row lane & 31 is unit K + 2 (lane >> 5), K = 8
    // pp + 4 hi + j, at byte 256 row + 16 ((K ^ 2 (lane >> 5)) ^ aswz(row))
    const uint32_t trd = 128u * row + 16u * (aswz(row) ^ (2 * half));
    const uint8_t *const tok = reinterpret_cast<const uint8_t *>(L.tok);
    uint32_t ml = 0x000f000fu, mh = 0x00f000f0u;
    asm volatile("" : "+s"(ml), "+s"(mh));
    const uint32_t ex = opaque(0x64006400u);
    __syncthreads();
    for (int sb = 0; sb < nsb; sb++) {
        if ((sb & 3) == 0 && sb) {
            uint4 r[2];
            hld(r, sb);
            hput(r);
        }
        const uint4 h = *reinterpret_cast<const uint4 *>(wh + (hrd ^ (16u * (sb & 3))));
        const float d = f16_bits_to_f32(h.x), dmin = f16_bits_to_f32(h.x >> 16);
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const int st = 4 * sb + p;
            const uint4 q = *reinterpret_cast<const uint4 *>(wq + (opaque(qrd) ^ (32u * p)));
            if (p == 3) {  // the super-block has been read: the next one in its place
                qput();
                qld(sb + 2);
            }
            awr(A[(p + 1) & 1], (p + 1) & 1);  // (past the end: a buffer nobody reads any more)
            ald(A[(p + 1) & 1], st + 3);
            const uint32_t tb = opaque(trd);
            // get_scale_min_k4 of sub-blocks 2 p, 2 p + 1
            const uint32_t ys = h.y >> (16 * (p & 1)), zs = h.z >> (16 * (p & 1)), ws = h.w >> (16 * (p & 1));
            const uint32_t scp = opaque(p < 2 ? (ys & 0x3f3fu) : ((ws & 0x0f0fu) | ((ys >> 2) & 0x3030u)));
            const uint32_t mnp = opaque(p < 2 ? (zs & 0x3f3fu) : (((ws >> 4) & 0x0f0fu) | ((zs >> 2) & 0x3030u)));
            const _Float16 d1 = (_Float16)(d * (float)(scp & 0xffu));
            const _Float16 m1 = (_Float16)(-(dmin * (float)(mnp & 0xffu)));
            const _Float16 d2 = (_Float16)(d * (float)((scp >> 8) & 0xffu) * 0.0625f);
            const _Float16 m2 = (_Float16)(-(dmin * (float)((mnp >> 8) & 0xffu)));
            const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
            for (int f = 0; f < 4; f++) {  // 2 hi + j
                f16x8 a[MT];
#pragma unroll
                for (int t = 0; t < MT; t++)
                    a[t] = *reinterpret_cast<const f16x8 *>(tok + (tb ^ (16u * (4 * (f >> 1) + (f & 1)))) +
                                                            2 * ((p & 1) * TB + t * 32 * KS));
                const uint32_t w0 = qw[2 * (f & 1)], w1 = qw[2 * (f & 1) + 1], m = f < 2 ? ml : mh;
                const half2v sc = f < 2 ? half2v{d1, d1} : half2v{d2, d2};
                const half2v nm = f < 2 ? half2v{m1, m1} : half2v{m2, m2};
                const f16x8 b =
                    q4_frag((w0 & m) | ex, ((w0 >> 8) & m) | ex, (w1 & m) | ex, ((w1 >> 8) & m) | ex, sc, nm);
#pragma unroll
                for (int t = 0; t < MT; t++)
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[t], b, acc[t], 0, 0, 0);
            }
            __syncthreads();
        }
    }
}

}  // namespace

// ---------------------------------------------------------------- dispatch
// Lanes of m below this lane.
__device__ __forceinline__ int rank_in(uint64_t m) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Block e places expert e's assignments: assignment i = t k + s goes to sorted
// row (number of valid ids below e) + (number of assignments before i with
// the same expert), a stable counting sort, so every row's chunk is the same
// on every call.  Wavefront w takes assignments [w seg, (w + 1) seg), 64 at a
// time: the lanes that hold e find their ranks with one ballot, and the
// wavefronts' totals meet in LDS.  Every block counts all experts as well (LDS
// atomics; a token's k experts are distinct, so few lanes share a counter),
// because a chunk's place in the list depends on all of them: full chunks in
// expert order first, then the partial ones of two token tiles, then of one
// -- the blocks with the most MFMA work are dispatched first and the short
// ones fill in behind them.  Each wavefront sums the counters for itself, so
// the counters' barrier is the only one behind the loads.  Up to kIds ids per
// lane are loaded once, all in flight together; longer batches read them
// again.
// Bound: the latency of the chain ids -> counters -> sums -> rows.  One block
// that sorted for all experts (a table of group sizes per 64 assignments and
// expert) took 6.4, 10.6 and 15.6 us for 37, 512 and 1024 tokens of 8 experts
// each out of 128, a block per expert 4.6, 7.0 and 10.2 us.
__global__ void __launch_bounds__(512) k_prefill_dispatch(const uint32_t *__restrict__ ids, int TK, int k, int E,
                                                          int *__restrict__ chunks, int *__restrict__ n_chunks,
                                                          int *__restrict__ perm, int *__restrict__ pos,
                                                          int *__restrict__ done, int maxc) {
    constexpr int kIds = 16, kWaves = 8;
    __shared__ int cnt[1024], own[kWaves];
    const int e = blockIdx.x, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int seg = (TK + 64 * kWaves - 1) / (64 * kWaves) * 64;
    const int i0 = wave * seg + lane, nj = seg / 64;  // this lane's assignments: i0 + 64 j, j < nj
    const bool cached = nj <= kIds;
    // i / k = i per_k / 2^31 for the i < 2^20 and k <= 16 there are: per_k k - 2^31 < k, and i k < 2^31
    const uint32_t per_k = ((1u << 31) + (uint32_t)k - 1) / (uint32_t)k;
    uint32_t xc[kIds];
    if (cached) {
#pragma unroll
        for (int j = 0; j < kIds; j++) xc[j] = j < nj && i0 + 64 * j < TK ? ids[i0 + 64 * j] : 0xffffffffu;
    }
    for (int q = tid; q < E; q += 512) cnt[q] = 0;
    for (int i = e * 512 + tid; i < maxc; i += 512 * E) done[i] = 0;  // the fused GEMMs' per-chunk counts
    __syncthreads();
    int mine = 0;  // (the wavefront's)
    auto count = [&](uint32_t x) {
        if (x < (uint32_t)E) atomicAdd(&cnt[x], 1);
        mine += __popcll(__ballot(x == (uint32_t)e));
    };
    if (cached) {
#pragma unroll
        for (int j = 0; j < kIds; j++)
            if (j < nj) count(xc[j]);
    } else {
#pragma unroll 8
        for (int j = 0; j < nj; j++) count(i0 + 64 * j < TK ? ids[i0 + 64 * j] : 0xffffffffu);
    }
    if (lane == 0) own[wave] = mine;
    __syncthreads();
    // rows below e, and the chunks of each kind (full, partial of two tiles, of
    // one): those below e in the low half, all of them in the high half
    int rows = 0, full = 0, two = 0, one = 0;
    for (int q = lane; q < E; q += 64) {
        const int n = cnt[q], rem = n % MC, f = q < e ? 0x10001 : 0x10000;
        rows += q < e ? n : 0;
        full += n / MC * f;
        two += rem > 32 ? f : 0;
        one += rem > 0 && rem <= 32 ? f : 0;
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        rows += __shfl_xor(rows, d, 64);
        full += __shfl_xor(full, d, 64);
        two += __shfl_xor(two, d, 64);
        one += __shfl_xor(one, d, 64);
    }
    const int tot_full = full >> 16, tot_two = two >> 16, n = cnt[e], nf = n / MC, rem = n % MC;
    if (e == 0 && tid == 0) *n_chunks = tot_full + tot_two + (one >> 16);
    // The list's places go round the 8 XCDs, so full chunk f of 8 q (the rest
    // at its own place) stands q places on in its XCD's row: the chunks of
    // one expert run beside each other on one XCD, whose L2 then holds the
    // weights they share (512 tokens 133.4 -> 131.6 us a call, 1024 209.3 -> 206.1).
    const int per = tot_full / 8;
    auto full_at = [&](int f) { return f < 8 * per ? f % per * 8 + f / per : f; };
    for (int c = tid; c < nf + (rem ? 1 : 0); c += 512) {
        const int at = c < nf      ? full_at((full & 0xffff) + c)
                       : rem > 32 ? tot_full + (two & 0xffff)
                                  : tot_full + tot_two + (one & 0xffff);
        chunks[3 * at] = e;
        chunks[3 * at + 1] = rows + c * MC;
        chunks[3 * at + 2] = c < nf ? MC : rem;
    }
    int row = rows;
#pragma unroll
    for (int w = 0; w < kWaves; w++) row += w < wave ? own[w] : 0;
    auto place = [&](uint32_t x, int i) {
        const uint64_t m = __ballot(x == (uint32_t)e);
        if (x == (uint32_t)e) {
            const int p = row + rank_in(m);
            perm[p] = (int)((uint64_t)i * per_k >> 31);
            pos[i] = p;
        } else if (e == 0 && x >= (uint32_t)E && i < TK) {
            pos[i] = -1;  // (no expert: the combine leaves the slot out)
        }
        row += __popcll(m);
    };
    if (cached) {
#pragma unroll
        for (int j = 0; j < kIds; j++)
            if (j < nj) place(xc[j], i0 + 64 * j);
    } else {
#pragma unroll 8
        for (int j = 0; j < nj; j++) place(i0 + 64 * j < TK ? ids[i0 + 64 * j] : 0xffffffffu, i0 + 64 * j);
    }
}

// X (fp32) -> f16, one block per token row (prefill_x_exp, prefill_x_store8:
// the row divided by rs = 2^e, stored in kperm order), for the router paths
// that do not write it themselves.  D % 8 == 0; the fp32 row is read twice
// (max, then values).
__global__ void __launch_bounds__(256) k_prefill_x_f16(const float *__restrict__ X, _Float16 *__restrict__ Xh,
                                                       float *__restrict__ rs, int D) {
    const int t = blockIdx.x, tid = threadIdx.x;
    const float *xr = X + (size_t)t * D;
    float m = 0.0f;
    for (int i = 4 * tid; i < D; i += 4 * 256) {
        const float4 v = ldg16f(xr + i);
        m = fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    }
    __shared__ float s_m[4];
    m = fmaxf(m, __shfl_xor(m, 32, 64));
    m = fmaxf(m, __shfl_xor(m, 16, 64));
    m = fmaxf(m, __shfl_xor(m, 8, 64));
    m = fmaxf(m, __shfl_xor(m, 4, 64));
    m = fmaxf(m, __shfl_xor(m, 2, 64));
    m = fmaxf(m, __shfl_xor(m, 1, 64));
    if ((tid & 63) == 0) s_m[tid >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(s_m[0], s_m[1]), fmaxf(s_m[2], s_m[3]));
    const int e = prefill_x_exp(m);
    const float inv = ldexpf(1.0f, -e);
    if (tid == 0) rs[t] = ldexpf(1.0f, e);
    _Float16 *hr = Xh + (size_t)t * D;
    for (int i = 8 * tid; i < D; i += 8 * 256) prefill_x_store8(xr, inv, hr, i);
}

// ---------------------------------------------------------------- gate/up
// The activation for the f16 H, branch-free: e^x and 1 / x as one hardware
// instruction each (v_exp_f32 on x log2 e, v_rcp_f32; about 1 ulp of fp32,
// far below the f16 rounding of H that follows).  SiLU g / (1 + e^-g);
// GELU (tanh form) 0.5 g (1 + tanh y) with tanh y = 1 - 2 / (1 + e^2y).
// Limits: g -> -inf gives -0 (SiLU) or 0, +inf gives g; NaN passes.
template <int ACT>
__device__ __forceinline__ float prefill_act(float g) {
    constexpr float kLog2e = 1.4426950408889634f;
    if (ACT == 1) {
        const float y = 0.7978845608028654f * (g + 0.044715f * g * g * g);
        const float t = 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(2.0f * kLog2e * y));
        return 0.5f * g * (1.0f + t);
    }
    return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-kLog2e * g));
}

namespace {

// Arguments of both grouped GEMMs (shared by their separate kernels and the
// fused one).
struct PfArgs {
    const uint8_t *gu_hdr, *gu_qs;  // gate/up planes: [E][2F] rows of gu_nsb super-blocks
    int gu_nsb, F;
    const _Float16 *Xh;
    const float *rs;
    int D;
    const int *chunks, *n_chunks, *perm;
    _Float16 *H;
    int Kd;
    const uint8_t *dn_hdr, *dn_qs;  // down planes: [E][D] rows of dn_nsb super-blocks
    int dn_nsb;
    float *Y;
    uint32_t *err;
    int *done;  // fused kernel: finished gate/up blocks per chunk (zeroed by the dispatch)
    int CG;     // fused kernel: chunk slots per XCD group
    const float *X;  // the fp32 input rows (one-token chunks)
    int tiny;        // one-token chunks take the decode-style stream (gate/up rows <= 8, down rows <= 4 super-blocks)
};

// ---------------------------------------------------------------- chunks of one token
// A chunk of one token streams its weights like the decode path instead of
// dequantising them to f16 tiles for a 32-row MFMA: the f16 tile costs the
// same whatever the chunk's rows, and many one-tile chunks of a skewed
// routing hold a single token (22 of the 63 in a 512-token batch with
// Zipf-biased logits).  (NT = 2 as well needed more registers than two
// waves per SIMD allow.)  A lane owns one Q4_K sub-block pair window
// (position 4 sb + p of a row: K elements 256 sb + 64 p + [0, 64)),
// whose activations it turns into int8 limbs in registers once (limbs16);
// per row it loads the window's 32 quant bytes and its quad's header word
// and meets them with each token's limbs on v_dot4 (q4k_pair_dot); a row's
// window dots meet in LDS and one lane adds them in position order, so
// results do not depend on timing.

struct WinW {
    uint4 q0, q1;
    uint32_t h;
};

__device__ __forceinline__ WinW load_window(const uint8_t *hdr, const uint8_t *qs, size_t blk, int p) {
    WinW w;
    w.q0 = ldg16(qs + blk * 128 + 32 * p);
    w.q1 = ldg16(qs + blk * 128 + 32 * p + 16);
    w.h = *reinterpret_cast<const uint32_t *>(hdr + blk * 16 + 4 * p);
    return w;
}

__device__ __forceinline__ float window_dot(const WinW &w, int p, const Limbs &xl) {
    uint32_t h0, h1, h2, h3;
    quad_header(w.h, h0, h1, h2, h3);
    const PairScale ps = pair_scale(h0, h1, h2, h3, p);
    const uint32_t w8[8] = {w.q0.x, w.q0.y, w.q0.z, w.q0.w, w.q1.x, w.q1.y, w.q1.z, w.q1.w};
    return q4k_pair_dot(w8, ps, xl);
}

// Gate/up of a chunk of NT tokens (one in use), columns n0 + [0, 64): wavefront
// w takes columns n0 + 16 w + c, one per pass c; lanes 0-31 the gate row,
// 32-63 the up row, lane l & 31 = window position (rows of at most 8
// super-blocks).  Weights two passes ahead; each lane's window dots go to
// LDS (red: [wave][pass][token][lane], the f16 tile's space) and lane c +
// 16 t + 32 half sums the 32 positions of (pass c, token t, gate or up) in
// position order.
template <int ACT, int NT>
__device__ __forceinline__ uint32_t gate_up_tiny(const PfArgs &a, float *red, const int *prow, int e, int row0,
                                                 int col0, int wave, int lane) {
    const int F = a.F, nsb = a.gu_nsb, Kd = a.Kd;
    const int pos = lane & 31, sb = min(pos >> 2, nsb - 1), p = pos & 3;
    const bool on = (pos >> 2) < nsb;
    const int half = lane >> 5;
    Limbs xl[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const float *xr = a.X + (size_t)prow[t] * a.D + 256 * sb + 64 * p;
        float xs[4];
#pragma unroll
        for (int g = 0; g < 4; g++) {  // group by group: 16 values live at a time
            float v[16];
#pragma unroll
            for (int i = 0; i < 16; i += 4) {
                const float4 f = ldg16f(xr + 16 * g + i);
                v[i] = f.x; v[i + 1] = f.y; v[i + 2] = f.z; v[i + 3] = f.w;
            }
            limbs16(v, xl[t].a[g], xl[t].b[g], xl[t].sp[g], xs[g]);
        }
        xl[t].xs_lo = xs[0] + xs[1];
        xl[t].xs_hi = xs[2] + xs[3];
    }
    auto blk_of = [&](int c) {
        const int col = col0 + c;
        return ((size_t)e * 2 * F + (half ? F + col : col)) * nsb + sb;
    };
    WinW w[16];
#pragma unroll
    for (int c = 0; c < 2; c++) w[c] = load_window(a.gu_hdr, a.gu_qs, blk_of(c), p);
    float *rw = red + wave * (16 * NT * 64);
#pragma unroll
    for (int c = 0; c < 16; c++) {
        if (c + 2 < 16) w[c + 2] = load_window(a.gu_hdr, a.gu_qs, blk_of(c + 2), p);
#pragma unroll
        for (int t = 0; t < NT; t++) rw[(c * NT + t) * 64 + lane] = on ? window_dot(w[c], p, xl[t]) : 0.0f;
    }
    __syncthreads();
    const int c = lane & 15, t = (lane >> 4) & 1;
    float v = 0.0f;
    if (t < NT) {
        const float *src = rw + (c * NT + t) * 64 + 32 * half;
#pragma unroll
        for (int q = 0; q < 32; q++) v += src[q];
    }
    const float up = __shfl(v, lane + 32, 64);  // (lanes 0-31: the up row's sum)
    uint32_t sat = 0;
    if (!half && t < NT) {
        // H = act(gate) * up / r^2 (r = 2^k exactly)
        const float r = a.rs[prow[t]];
        const float ri = __builtin_amdgcn_ldexpf(1.0f, 1 - __builtin_amdgcn_frexp_expf(r));
        const float h = prefill_act<ACT>(v) * up * ri * ri;
        const bool big = fabsf(h) > 65504.0f && fabsf(h) <= 3.4e38f;
        sat = big ? 1u : 0u;
        a.H[(size_t)(row0 + t) * Kd + kperm(col0 + c)] = (_Float16)(big ? copysignf(65504.0f, h) : h);
    }
    return sat;
}

// Down of a chunk of NT tokens (one in use), output rows n0 + [0, 128): lanes
// l & 15 = window position (K of at most 4 super-blocks), lane >> 4 = row
// of the pass; wavefront w takes rows n0 + 32 w + 4 c + (lane >> 4), pass
// c < 8.  The activations are the H rows (f16, K in kperm order).  Lane
// c + 8 rr + 32 t then sums the 16 positions of (pass c, row rr, token t).
template <int NT, typename Wait>
__device__ __forceinline__ void down_tiny(const PfArgs &a, float *red, int e, int row0, int nrow, Wait wait, int wave,
                                          int lane) {
    const int nsb = a.dn_nsb, D = a.D, Kd = a.Kd;
    const int pos = lane & 15, sb = min(pos >> 2, nsb - 1), p = pos & 3;
    const bool on = (pos >> 2) < nsb;
    const int rr = lane >> 4;
    auto blk_of = [&](int c) { return ((size_t)e * D + nrow + 4 * c + rr) * nsb + sb; };
    WinW w[8];
#pragma unroll
    for (int c = 0; c < 2; c++) w[c] = load_window(a.dn_hdr, a.dn_qs, blk_of(c), p);
    wait();
    Limbs xl[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const _Float16 *hr = a.H + (size_t)(row0 + t) * Kd + 256 * sb + 64 * p;
        float xs[4];
#pragma unroll
        for (int g = 0; g < 4; g++) {  // group by group: 16 values live at a time
            float v[16];
#pragma unroll
            for (int i = 0; i < 16; i += 8) {
                const uint4 u = *reinterpret_cast<const uint4 *>(hr + 16 * g + i);  // h[kperm(.. + j)], j < 8
                const uint32_t wd[4] = {u.x, u.y, u.z, u.w};
                _Float16 f[8];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    f[2 * j] = __builtin_bit_cast(_Float16, (uint16_t)(wd[j] & 0xffffu));
                    f[2 * j + 1] = __builtin_bit_cast(_Float16, (uint16_t)(wd[j] >> 16));
                }
#pragma unroll
                for (int j = 0; j < 8; j++) v[i + kperm(j)] = (float)f[j];
            }
            limbs16(v, xl[t].a[g], xl[t].b[g], xl[t].sp[g], xs[g]);
        }
        xl[t].xs_lo = xs[0] + xs[1];
        xl[t].xs_hi = xs[2] + xs[3];
    }
    float *rw = red + wave * (8 * NT * 64);
#pragma unroll
    for (int c = 0; c < 8; c++) {
        if (c + 2 < 8) w[c + 2] = load_window(a.dn_hdr, a.dn_qs, blk_of(c + 2), p);
#pragma unroll
        for (int t = 0; t < NT; t++) rw[(c * NT + t) * 64 + lane] = on ? window_dot(w[c], p, xl[t]) : 0.0f;
    }
    __syncthreads();
    const int c = lane & 7, r4 = (lane >> 3) & 3, t = lane >> 5;
    if (t < NT) {
        const float *src = rw + (c * NT + t) * 64 + 16 * r4;
        float v = 0.0f;
#pragma unroll
        for (int q = 0; q < 16; q++) v += src[q];
        a.Y[(size_t)(row0 + t) * D + nrow + 4 * c + r4] = v;
    }
}

// acc element i of a 32 x 32 tile is C[tile_row(i, lane)][lane & 31].
__device__ __forceinline__ int tile_row(int i, int lane) { return (i >> 2) * 8 + (lane >> 5) * 4 + (i & 3); }

// The tiles of a gate/up block: wavefront w has gate columns n0 + 16 w + [0,
// 16) in its rows 0-15 and the matching up columns in rows 16-31.  The halves
// trade values (element i's up against element i + 1's gate), so that lanes
// 0-15 of a 32-lane half finish element i and lanes 16-31 element i + 1.
// With r the token's row scale, gate = r g and up = r u, and H = act(gate) *
// up / r^2 = act(r g) * (u / r) (exact scalings), stored in kperm order (the
// down GEMM's K); a finite value past f16's range saturates at +-65504 and is
// counted (inf and NaN pass through).
template <int ACT, int MT>
__device__ __forceinline__ uint32_t gate_up_tiles(const PfArgs &a, GemmLds &L, const int *prow, size_t wrow0, int row0,
                                                  int mc, int col, int wave, int tid, int lane) {
    floatx16 acc[MT];
    uint32_t aoff[MT];
    const float rt = a.rs[prow[tid < mc ? tid : 0]];  // (rows past the chunk repeat its first one)
#pragma unroll
    for (int t = 0; t < MT; t++) {
        const int m = 32 * t + (tid >> 3);
        aoff[t] = (uint32_t)prow[m < mc ? m : 0] * (uint32_t)(a.D / 8) + (tid & 7);
    }
    gemm_tiles<MT>(acc, L, a.gu_hdr + wrow0 * a.gu_nsb * 16, a.gu_qs + wrow0 * a.gu_nsb * 128, (uint32_t)a.F,
                   a.gu_nsb, reinterpret_cast<const uint8_t *>(a.Xh), aoff, wave, tid, lane, NoWait{});
    // row scales r and 1 / r (r = 2^k exactly: frexp gives k + 1, so 1 / r = 2^(1 - (k + 1)))
    float2 *const rs = reinterpret_cast<float2 *>(L.tok);  // (free behind the GEMM's last barrier)
    if (tid < MC) rs[tid] = make_float2(rt, __builtin_amdgcn_ldexpf(1.0f, 1 - __builtin_amdgcn_frexp_expf(rt)));
    __syncthreads();
    // The block's H tile, 64 columns (128 bytes) a row, goes out through LDS in
    // 16-byte stores.
    uint32_t sat = 0;
    const int up1 = (lane >> 4) & 1;
    _Float16 *const ht = reinterpret_cast<_Float16 *>(L.tok) + 4 * MC + kperm(16 * wave + (lane & 15));
    float top = 0.0f;
    auto tile = [&](auto put) {
#pragma unroll
        for (int t = 0; t < MT; t++) {
#pragma unroll
            for (int i = 0; i < 16; i += 2) {
                const float other = xor16(up1 ? acc[t][i] : acc[t][i + 1]);
                const float g = up1 ? other : acc[t][i], u = up1 ? acc[t][i + 1] : other;
                const int m = 32 * t + tile_row(i, lane) + up1;
                const float2 r = rs[m];
                put(m, prefill_act<ACT>(g * r.x) * (u * r.y));
            }
        }
    };
    tile([&](int m, float h) {
        top = fmaxf(top, fabsf(h));
        ht[BN1 * m] = (_Float16)h;
    });
    // (rare: rows in range and finite values saturate and count, inf and NaN
    // stay; the whole wavefront goes, as each element needs its partner lane's half)
    if (__any(top > 65504.0f))
        tile([&](int m, float h) {
            const bool big = fabsf(h) > 65504.0f && fabsf(h) <= 3.4e38f;
            sat += big && m < mc ? 1u : 0u;
            ht[BN1 * m] = (_Float16)(big ? copysignf(65504.0f, h) : h);
        });
    __syncthreads();
    const int un = tid & 7;
    _Float16 *const hout = a.H + (size_t)row0 * a.Kd + (col - 16 * wave) + 8 * un;
#pragma unroll
    for (int t = 0; t < MT; t++) {
        const int m = 32 * t + (tid >> 3);
        if (m < mc)
            *reinterpret_cast<uint4 *>(hout + (size_t)m * (uint32_t)a.Kd) =
                *reinterpret_cast<const uint4 *>(L.tok + 4 * MC + BN1 * m + 8 * un);
    }
    return sat;
}

// Block: chunk (expert e, sorted rows row0 + [0, mc)) x output columns n0 +
// [0, 64).  ACT: the activation (0 SiLU, 1 GELU-tanh).  False when the
// chunk does not exist.
template <int ACT>
__device__ __forceinline__ bool gate_up_body(const PfArgs &a, int bx, int by, GemmLds &L) {
    if (by >= *a.n_chunks) return false;
    const int e = __builtin_amdgcn_readfirstlane(a.chunks[3 * by]);
    const int mc = __builtin_amdgcn_readfirstlane(a.chunks[3 * by + 2]);
    const int row0 = __builtin_amdgcn_readfirstlane(a.chunks[3 * by + 1]);
    const int n0 = bx * BN1, F = a.F, Kd = a.Kd;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int col = n0 + 16 * wave;  // this wavefront's 16 columns (F % 64 == 0)
    const int *prow = a.perm + row0;
    uint32_t sat = 0;
    if (a.tiny && mc == 1) {
        sat = gate_up_tiny<ACT, 1>(a, reinterpret_cast<float *>(L.tok), prow, e, row0, col, wave, lane);
    } else {
        // rows 8 j + (lane >> 3) of the wavefront: gate columns for j < 2, up columns for the others
        const size_t wrow0 = (size_t)e * 2 * F + col;
        sat = mc <= 32 ? gate_up_tiles<ACT, 1>(a, L, prow, wrow0, row0, mc, col, wave, tid, lane)
                       : gate_up_tiles<ACT, 2>(a, L, prow, wrow0, row0, mc, col, wave, tid, lane);
    }
    if (sat) {  // (rare): the count and the error bit, reported at the next synchronising call
        __hip_atomic_fetch_add(a.err + kErrPrefillSat, sat, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        report_timeout(a.err, kErrCodePrefillSat);
    }
    if (bx == 0 && Kd > F)  // zero K padding of the down product
        for (int i = tid; i < mc * (Kd - F); i += PT) {
            const int m = i / (Kd - F), c = F + i % (Kd - F);
            a.H[(size_t)(row0 + m) * Kd + c] = (_Float16)0.f;  // (kperm keeps [F, Kd): F % 4 == 0)
        }
    return true;
}

template <int MT, typename Wait>
__device__ __forceinline__ void down_tiles(const PfArgs &a, GemmLds &L, size_t wrow0, int row0, int mc, int n, Wait wait,
                                           int wave, int tid, int lane) {
    floatx16 acc[MT];
    uint32_t aoff[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) {
        const int m = 32 * t + (tid >> 3);
        aoff[t] = (uint32_t)(m < mc ? m : 0) * (uint32_t)(a.Kd / 8) + (tid & 7);
    }
    gemm_tiles<MT>(acc, L, a.dn_hdr + wrow0 * a.dn_nsb * 16, a.dn_qs + wrow0 * a.dn_nsb * 128, 16u, a.dn_nsb,
                   reinterpret_cast<const uint8_t *>(a.H + (size_t)row0 * a.Kd), aoff, wave, tid, lane, wait);
    float *ycol = a.Y + (size_t)row0 * a.D + n + (lane & 31);
#pragma unroll
    for (int t = 0; t < MT; t++) {
        const bool full = 32 * t + 32 <= mc;  // (uniform: no branch per element)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int m = 32 * t + tile_row(i, lane);
            if (full || m < mc) ycol[(size_t)m * (uint32_t)a.D] = acc[t][i];
        }
    }
}

// Block: chunk x output rows n0 + [0, 128) of the expert's down matrix (=
// columns of Y), 32 a wavefront; the token operand is the H rows (f16).
template <typename Wait>
__device__ __forceinline__ void down_body(const PfArgs &a, int bx, int by, GemmLds &L, Wait wait) {
    const int e = __builtin_amdgcn_readfirstlane(a.chunks[3 * by]);
    const int mc = __builtin_amdgcn_readfirstlane(a.chunks[3 * by + 2]);
    const int row0 = __builtin_amdgcn_readfirstlane(a.chunks[3 * by + 1]);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int n = bx * BN2 + 32 * wave;  // (D % 128 == 0)
    if (a.tiny && mc == 1) {
        down_tiny<1>(a, reinterpret_cast<float *>(L.tok), e, row0, n, wait, wave, lane);
        return;
    }
    const size_t wrow0 = (size_t)e * a.D + n;
    if (mc <= 32)
        down_tiles<1>(a, L, wrow0, row0, mc, n, wait, wave, tid, lane);
    else
        down_tiles<2>(a, L, wrow0, row0, mc, n, wait, wave, tid, lane);
}

constexpr uint64_t kPfWaitTicks = 20000000;  // 200 ms of the 100 MHz wall clock

}  // namespace

template <int ACT>
__global__ void __launch_bounds__(PT, 4) k_prefill_gate_up(PfArgs a) {
    __shared__ GemmLds L;
    gate_up_body<ACT>(a, blockIdx.x, blockIdx.y, L);
}

// ---------------------------------------------------------------- down
__global__ void __launch_bounds__(PT, 4) k_prefill_down(PfArgs a) {
    if ((int)blockIdx.y >= *a.n_chunks) return;
    __shared__ GemmLds L;
    down_body(a, blockIdx.x, blockIdx.y, L, NoWait{});
}

// ---------------------------------------------------------------- both GEMMs in one launch
// Block b of XCD group g = b % 8 (blocks with equal b % 8 share an XCD, as
// probed once per context), in-group index s = b / 8: the first
// (F / 64) CG indices are the gate/up blocks of the group's chunks
// y = g + 8c (c = s / (F / 64), column block s % (F / 64)), the next
// (D / 128) CG the down blocks of the same chunks, in the same chunk order.
// A gate/up block's H rows are ordinary stores that stay in its XCD's L2;
// once they are acknowledged it adds 1 to done[y].  A down block requests
// its first weight stages, then waits until done[y] = F / 64 and reads H
// through the same L2.  So the down blocks of the first chunks run while
// the last gate/up blocks finish, instead of behind the whole gate/up grid.
// A down block only waits for blocks with smaller indices, which are
// dispatched first; the wait is bounded by the wall clock (on expiry the
// error word is set and that call's outputs are wrong).
template <int ACT>
__global__ void __launch_bounds__(PT, 4) k_prefill_gemms(PfArgs a) {
    __shared__ GemmLds L;
    const int g = blockIdx.x & 7, s = blockIdx.x >> 3;
    const int ngx = a.F / BN1, ngu = ngx * a.CG;
    if (s < ngu) {
        const int y = g + 8 * (s / ngx);
        if (!gate_up_body<ACT>(a, s % ngx, y, L)) return;
        // every thread's H stores acknowledged by the L2 before the count
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) __hip_atomic_fetch_add(a.done + y, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    const int ndx = a.D / BN2, s2 = s - ngu;
    const int y = g + 8 * (s2 / ndx);
    if (y >= *a.n_chunks) return;
    auto wait = [&] {
        if (threadIdx.x == 0) {
            const uint64_t t0 = wall_clock64();
            int seen;
            while ((seen = __hip_atomic_load(a.done + y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) < ngx) {
                if (wall_clock64() - t0 > kPfWaitTicks) {
                    report_timeout(a.err, kErrCodePrefillWait);
                    report_detail(a.err, (int)blockIdx.x, kErrCodePrefillWait, (uint32_t)y, (uint32_t)seen,
                                  (uint32_t)ngx);
                    break;
                }
                __builtin_amdgcn_s_sleep(2);
            }
        }
        __syncthreads();
    };
    down_body(a, s2 % ndx, y, L, wait);
}

// ---------------------------------------------------------------- combine
// Thread: 4 consecutive elements of one token's row (D % 4 == 0); every
// slot's Y row is read with one 16-byte load per thread, all k loads in
// flight before the sum, which runs in slot order; the sum times r_t^2
// (the row scale the activations were divided by, exact).
__global__ void __launch_bounds__(256) k_prefill_combine(const float *__restrict__ Y, const int *__restrict__ pos,
                                                         const float *__restrict__ w, const float *__restrict__ rs,
                                                         int k, int D, float *__restrict__ out) {
    const int t = blockIdx.y, i = 4 * (blockIdx.x * 256 + threadIdx.x);
    if (i >= D) return;
    float4 v[16];
    float ws[16];
#pragma unroll
    for (int s = 0; s < 16; s++) {
        if (s < k) {
            const int p = pos[t * k + s];
            ws[s] = p >= 0 ? w[t * k + s] : 0.0f;
            v[s] = ldg16f(Y + (size_t)(p >= 0 ? p : 0) * D + i);
        }
    }
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int s = 0; s < 16; s++) {
        if (s < k && pos[t * k + s] >= 0) {
            acc.x += ws[s] * v[s].x;
            acc.y += ws[s] * v[s].y;
            acc.z += ws[s] * v[s].z;
            acc.w += ws[s] * v[s].w;
        }
    }
    const float r2 = rs[t] * rs[t];
    acc.x *= r2;
    acc.y *= r2;
    acc.z *= r2;
    acc.w *= r2;
    *reinterpret_cast<float4 *>(out + (size_t)t * D + i) = acc;
}

size_t prefill_workspace_bytes(int T, int k, int E, int Kd, int D) {
    const size_t TK = (size_t)T * k;
    return align256((size_t)T * E * 4) + 2 * align256(TK * 4) +
           align256((size_t)max_chunks((int)TK, E) * 12) + 256 + 2 * align256(TK * 4) + align256((size_t)T * 4) +
           align256((size_t)T * D * 2) + align256(TK * Kd * 2) + align256(TK * D * 4) +
           align256((size_t)max_chunks((int)TK, E) * 4);
}

hipError_t launch_moe_prefill(const DevTensor &R, const DevTensor &GU, const DevTensor &Dn, const float *X, int T,
                              const float *bias, int k, int F, uint32_t act, uint32_t norm, void *ws, float *out,
                              uint32_t *out_ids, float *out_w, uint32_t *err, int xcd_local, hipStream_t s) {
    const int E = (int)GU.n_experts, D = (int)GU.cols, Kd = (int)Dn.cols;
    const int TK = T * k;
    Ws w = carve(ws, T, k, E, Kd, D);
    bool x_done = false;
    hipError_t e = launch_router_batched(R, X, T, bias, w.logits, k, norm, w.ids, w.w, w.Xh, w.rs, &x_done, s);
    if (e != hipSuccess) return e;
    const int mc = max_chunks(TK, E);
    hipLaunchKernelGGL(k_prefill_dispatch, dim3(E), dim3(512), 0, s, w.ids, TK, k, E, w.chunks, w.n_chunks,
                       w.perm, w.pos, w.done, mc);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (!x_done) {
        hipLaunchKernelGGL(k_prefill_x_f16, dim3((unsigned)T), dim3(256), 0, s, X, w.Xh, w.rs, D);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    PfArgs pa{};
    pa.gu_hdr = (const uint8_t *)GU.p0;
    pa.gu_qs = (const uint8_t *)GU.p1;
    pa.gu_nsb = (int)GU.blocks_per_row;
    pa.F = F;
    pa.Xh = w.Xh;
    pa.rs = w.rs;
    pa.D = D;
    pa.chunks = w.chunks;
    pa.n_chunks = w.n_chunks;
    pa.perm = w.perm;
    pa.H = w.H;
    pa.Kd = Kd;
    pa.dn_hdr = (const uint8_t *)Dn.p0;
    pa.dn_qs = (const uint8_t *)Dn.p1;
    pa.dn_nsb = (int)Dn.blocks_per_row;
    pa.Y = w.Y;
    pa.err = err;
    pa.done = w.done;
    pa.CG = (mc + 7) / 8;
    pa.X = X;
    // (LT_PREFILL_NO_TINY, read at each call: every chunk on the tiles, for testing)
    pa.tiny = GU.blocks_per_row <= 8 && Dn.blocks_per_row <= 4 && !getenv("LT_PREFILL_NO_TINY");
    const int ngx = F / BN1, ndx = D / BN2;
    if (xcd_local) {
        // Blocks a CU: four, or two (16 KB more LDS a block) where the gate/up
        // blocks to be expected -- a chunk per MC rows and one more for half
        // of the experts -- leave places free at four a CU.  Down blocks of
        // unfinished chunks would take those places, each fixed to the CU it
        // waits on, and what they then draw from memory delays the gate/up
        // blocks beside them that others still wait for.  Whole calls, four |
        // two a CU, 2048 x 768, 128 experts, 8 a token, routing as skewed as
        // a text's: 8 tokens 67 | 62 us, 37 92 | 71, 100 109 | 85, 200 101 |
        // 106, 512 143 | 161, 1024 219 | 242; 1000 tokens of 1280 x 448, 32
        // experts, 4 a token: 113 | 85.  (Even routings, with a chunk for
        // every expert, turn earlier: 64 tokens 108 | 121, 135 before 64-row
        // chunks, but the host does not know them.)
        const unsigned nb = 8u * (unsigned)((ngx + ndx) * pa.CG);
        const bool two = (TK / MC + min(E, TK) / 2) * ngx < 4 * 256;
        hipLaunchKernelGGL(act == 1u ? k_prefill_gemms<1> : k_prefill_gemms<0>, dim3(nb), dim3(PT), two ? 16384 : 0, s,
                           pa);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    } else {
        hipLaunchKernelGGL(act == 1u ? k_prefill_gate_up<1> : k_prefill_gate_up<0>, dim3(ngx, mc), dim3(PT), 0, s,
                           pa);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        hipLaunchKernelGGL(k_prefill_down, dim3(ndx, mc), dim3(PT), 0, s, pa);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_prefill_combine, dim3((D / 4 + 255) / 256, T), dim3(256), 0, s, w.Y, w.pos, w.w, w.rs, k, D,
                       out);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (out_ids) {
        if ((e = hipMemcpyAsync(out_ids, w.ids, (size_t)TK * 4, hipMemcpyDefault, s)) != hipSuccess) return e;
    }
    if (out_w) {
        if ((e = hipMemcpyAsync(out_w, w.w, (size_t)TK * 4, hipMemcpyDefault, s)) != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace lt
