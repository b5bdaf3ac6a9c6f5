// bruteforce_mfma.hip -- the screening pass of the exact k-nearest-neighbour search on the matrix cores.
//
// The exact search (bruteforce.hip) accumulates every (query, base) pair in the reference's order, one fused
// multiply-add per dimension on the vector units, because ids and distances must be reproducible bit for bit.  Almost
// all of that work goes into pairs that are nowhere near the k best.  Here the same pairs are first measured
// approximately, as |q|^2 + |b|^2 - 2 q.b with the inner products on the matrix cores, k + 32 candidates per query
// are kept, and rerank_kernel measures just those in the reference's order.  The result is exact, not approximately
// exact: a query is accepted only if its k-th exact distance lies below the worst kept approximate distance by more
// than a bound on what the two ways of rounding can differ by; otherwise it is flagged and goes through the exact
// search.
//
// The inner products: rows are split into two planes of halves (mfma_split.h, with the bound on what that and the
// accumulation lose), and q.b = hi.hi + hi.lo + lo.hi on v_mfma_f32_32x32x16_f16: three multiplications at sixteen
// times the rate of the fp32 form.
//
// Large batches are first screened on hi.hi alone, a third of the products.  No value of that screening goes anywhere
// but into the choice of candidates, and the choice stays rigorous: what the missing products amount to is bounded by
// |q - hi(q)| |b| + |hi(q)| |b - hi(b)| (row_norms_kernel measures both factors; about 3e-4 |q| |b|), the check
// below takes that much more, and queries that fail it go through the screening on three products.  k + 32 candidates
// leave room for the entries that one product cannot tell apart wherever distances spread by more than a few
// thousandths of |q| |b|; whether they do is read off the sample before the base is walked (count_close_kernel).
// 10 000 x 1 000 000 x 200, k = 100: 18.2 -> 12.0 ms.
//
// Error bound, with u = 2^-24 and n2 = |q|^2 + |b|^2.
// L2.  The inner product is within (6 dim + 12) u |q| |b| and enters twice: (6 dim + 12) u n2.  The two norms are within
// dim u of themselves, the final additions add 3 u n2, and terms of second order come to less than 14 u n2 at 2048
// dimensions: the approximate distance is within E = (7 dim + 32) u n2 of the true one.  The reference-order distance is
// within (dim + 2) u of the true one, relative to that.  So a point whose approximate distance is no less than `worst` has
// a reference-order distance of at least worst - E - (dim + 2) u worst; the check takes (dim + 8) u worst for the last
// term, which leaves room for its own rounding.
// Inner product.  (3 dim + 6) u n2 for the product, u n2 / 2 for the last rounding, dim u n2 / 2 for the reference order:
// the check takes 4 (dim + 8) u n2.
// Either way 2^-149 is added for each operation whose result may leave the normal range, 10 (dim + 4) of them (what the
// clamped scale of rows shorter than 2^-47 loses is less), and the largest |b|^2 of the index stands for |b|^2.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "bruteforce.h"
#include "mfma_split.h"

namespace coral {

namespace {

constexpr int kMatrix = 0, kFused = 1, kLevels = 2;  // what a launch of the tile kernel writes
constexpr int MT = 256, NT = 128, BK = 16;  // tile of queries x base points per workgroup, dimensions per LDS stage
constexpr int kStageA = 2 * MT * BK, kStageB = 2 * NT * BK;  // halves per stage: two planes
// NP: products per pair and dimension.  3: the planes are the hi and the lo halves of 16 dimensions; 1: the hi halves of
// 32 dimensions
template <int NP>
constexpr int kStageDims = NP == 1 ? 2 * BK : BK;

__device__ __forceinline__ uint32_t mf_ord32(float s) {
    const uint32_t u = __float_as_uint(s);
    return u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
}
__device__ __forceinline__ float mf_unord32(uint32_t o) {
    const uint32_t u = (o & 0x80000000u) ? (o ^ 0x80000000u) : ~o;
    return __uint_as_float(u);
}

// |x|^2 of a row, lane by lane side by side; in every lane
__device__ __forceinline__ float row_norm(const float4* __restrict__ p, int chunks, int lane) {
    float s = 0.0f;
    for (int c = lane; c < chunks; c += 64) {
        const float4 v = p[c];
        s = __fmaf_rn(v.x, v.x, s), s = __fmaf_rn(v.y, v.y, s), s = __fmaf_rn(v.z, v.z, s), s = __fmaf_rn(v.w, v.w, s);
    }
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    return s;
}

// a bound on what a row of squared norm s loses when each component of it, scaled as the tile kernel scales it, becomes one
// half: |x - half(x)|.  (Halves below the format's normal range count as lost whole, so the bound holds whether or not the
// matrix cores take them for zero.  A row of infinite or NaN norm gives an infinite or NaN bound, which no comparison passes.)
__device__ __forceinline__ float row_loss(const float4* __restrict__ p, int chunks, int lane, float s) {
    const int e = mf_scale_exp(s);
    const float up = mf_pow2(e);
    float l2 = 0.0f;
    for (int c = lane; c < chunks; c += 64) {
        const float4 v = p[c];
        const float w[4] = {v.x * up, v.y * up, v.z * up, v.w * up};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float h = (float)(_Float16)w[j];
            const float d = fabsf(h) < 6.2e-5f ? w[j] : w[j] - h;
            l2 = __fmaf_rn(d, d, l2);
        }
    }
    for (int off = 32; off > 0; off >>= 1) l2 += __shfl_xor(l2, off, 64);
    // (2^-51 <= 2^e <= 2^60; the sum of squares is within dim 2^-24 of itself; the last term for squares that leave the
    // normal range)
    const float lost = (sqrtf(l2) * (1.0f + 2.0e-4f) + 1.0e-17f) * mf_pow2(-e);
    return s <= 3.0e38f ? lost : __int_as_float(0x7f800000);
}

// |x|^2 per row, the largest of them (as the bit pattern of a non-negative float), and the largest loss.
// One wavefront per row.  (A thread per row read 16 bytes of a line at a time: the norms of 1M x 200 took 724 us, of a
// batch of 2000 x 512 as long as 45.  An atomic per wavefront of 8192 workgroups, all on one word, made 50 000 x 100 take 374.)
__global__ __launch_bounds__(256) void row_norms_kernel(const float* __restrict__ x, int64_t n, int dim,
                                                       float* __restrict__ out, uint32_t* __restrict__ max_bits,
                                                       uint32_t* __restrict__ res_max) {
    const int lane = threadIdx.x & 63, chunks = dim >> 2;
    const int64_t waves = (int64_t)gridDim.x * 4;
    float most = 0.0f, most_lost = 0.0f;
    for (int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); r < n; r += waves) {
        const float4* p = reinterpret_cast<const float4*>(x + (size_t)r * dim);
        const float s = row_norm(p, chunks, lane);
        if (out && lane == 0) out[r] = s;
        most = s > most ? s : (s != s ? s : most);  // (a NaN stays)
        if (res_max) most_lost = fmaxf(most_lost, row_loss(p, chunks, lane, s));
    }
    __shared__ uint32_t wave_most[4][2];
    if (lane == 0) wave_most[threadIdx.x >> 6][0] = __float_as_uint(most), wave_most[threadIdx.x >> 6][1] = __float_as_uint(most_lost);
    __syncthreads();
    if (threadIdx.x < 2) {
        uint32_t* to = threadIdx.x == 0 ? max_bits : res_max;
        const uint32_t m = max(max(wave_most[0][threadIdx.x], wave_most[1][threadIdx.x]),
                               max(wave_most[2][threadIdx.x], wave_most[3][threadIdx.x]));
        if (to && __hip_atomic_load(to, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < m) atomicMax(to, m);
    }
}

// The queries as the tile kernel reads them: per tile of 256 queries and stage, two planes of [256 rows][16 halves] --
// a stage of a tile is 16 KB in the order in which it lies in LDS.  NP = 3: the hi and the lo plane of 16 dimensions;
// NP = 1: the hi planes of 32.  Rows beyond the batch and dimensions beyond dim are zero.  On the way |q|^2 (and with res
// the bound on what one half per component leaves out), the query's counter and the two words of `zero` are set: what
// would be three launches more, each longer on its way to the chip than on it for a small batch.
// One wavefront per row, as row_norms_kernel reads it.
template <int NP>
__global__ __launch_bounds__(256) void prepare_queries_kernel(const float* __restrict__ queries, int nq, int dim, int stages,
                                                             float* __restrict__ qn, float* __restrict__ res,
                                                             _Float16* __restrict__ out, unsigned int* __restrict__ cnt,
                                                             int* __restrict__ zero) {
    const int lane = threadIdx.x & 63, chunks = dim >> 2;
    const int64_t q = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const float4* p = reinterpret_cast<const float4*>(queries + (size_t)q * dim);
    float s = 0.0f;
    if (q < nq) {
        s = row_norm(p, chunks, lane);
        const float lost = res ? row_loss(p, chunks, lane, s) : 0.0f;
        if (lane == 0) {
            qn[q] = s;
            if (res) res[q] = lost;
            if (cnt) cnt[(size_t)q * kCntStride] = 0u;
        }
    }
    if (zero && q == 0 && lane < 2) zero[lane] = 0;
    const float up = mf_pow2(mf_scale_exp(s));
    _Float16* tile = out + (size_t)(q / MT) * stages * kStageA + (q % MT) * BK;
    for (int c = lane; c < stages * (kStageDims<NP> / 4); c += 64) {
        const int k = 4 * c;
        float4 v = make_float4(0, 0, 0, 0);
        if (q < nq && k < dim) v = p[c];
        v4h hi, lo;
        mf_split4(v, up, hi, lo);
        _Float16* dst = tile + (size_t)(k / kStageDims<NP>) * kStageA + (k % kStageDims<NP>) / BK * (MT * BK) + k % BK;
        *reinterpret_cast<v4h*>(dst) = hi;
        if (NP == 3) *reinterpret_cast<v4h*>(dst + MT * BK) = lo;
    }
}

// D[q][b] ~ signed distance (smaller is closer): |q|^2 + |b|^2 - 2 q.b for L2, -q.b for IP; +inf for tombstoned
// ids.  One workgroup per 256 x 128 tile (the mapping of blockIdx to tiles is at the head of the kernel), 256
// threads = 4 wavefronts in 2 x 2, each 128 x 64 of the tile as 4 x 2 MFMA blocks of 32 x 32.
// MODE = kMatrix writes the tile into D (column bt * 128 + ..., where bt counts the tiles this launch computes).
// MODE = kLevels (NP = 1) writes four bits per entry: which of fifteen steps of the query's range (origin, step) the
// value falls into, 0 and 14 open to below and above, entries of rows whose norm is not finite or beyond 1e37 always 0;
// the matrix is computed with the operands exchanged, so that a lane holds four consecutive base points of one query and
// packs them by itself.  The tile's levels leave through LDS, 64 bytes per query.
// MODE = kFused writes no matrix: an entry goes, as the key ord(value) << 32 | id, to the list of its query if it does
// not exceed the query's bound tau[q] -- cnt[q * kCntStride] entries so far, at most cap kept (a count beyond cap
// tells the caller that the list is incomplete).  A tile's entries are first gathered in LDS, so that the global
// counters see one round of atomics per tile instead of one per accumulator register.
// The tiles of a launch: tile_step > 0 takes tiles 0, tile_step, 2 tile_step ... of the base, tile_step < 0 the tiles
// between those (all that are no multiple of -tile_step).
//
// Bound by the matrix cores in principle (three half-precision products per pair and dimension, 833 TFLOP/s of
// pair-dimensions at the card's dense rate), in practice by LDS: a wavefront reads 12 KB per 24 multiplications
// (768 cycles of its matrix core; the reads of a CU's four wavefronts take 384 cycles of its LDS, parking the next
// stage 192), which is why a wavefront has a 128 x 64 tile and not the 64 x 64 that the fp32 form had.  The queries
// come split (prepare_queries_kernel: every query tile is read by thousands of workgroups); the base is split here, on
// its way to LDS, eight components per thread and stage under the other wavefronts' multiplications: a split copy of
// the base would double the index or cost a pass over it per call, which small batches would feel.
template <int MODE, bool L2, int NP>
__global__ __launch_bounds__(256, 2) void approx_tile_mfma_kernel(const _Float16* __restrict__ queries,
                                                              const float* __restrict__ base, int nq, int64_t nb,
                                                              int dim, const float* __restrict__ qn,
                                                              const float* __restrict__ bn,
                                                              const uint32_t* __restrict__ deleted, int64_t base_id0,
                                                              int64_t ntiles, int tile_step, int hq,
                                                              float* __restrict__ D, int64_t ldD,
                                                              const float* __restrict__ tau,
                                                              unsigned long long* __restrict__ lists, int64_t cap,
                                                              unsigned int* __restrict__ cnt, const float4* __restrict__ ranges,
                                                              unsigned char* __restrict__ levels, size_t pitch) {
    constexpr bool FUSED = MODE == kFused;
    static_assert(MODE != kLevels || NP == 1, "levels are made on one product");
    // A row's 16 dimensions of a plane lie side by side (32 bytes); lane (kh, m) of a wavefront supplies row m's
    // dimensions kh * 8 .. + 7, one 16-byte read, and the 64 lanes of a read cover 2 KB of consecutive addresses.
    __shared__ __align__(16) _Float16 sa[2][kStageA];
    __shared__ __align__(16) _Float16 sb[2][kStageB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave >> 1, wc = wave & 1;
    // Workgroups go to the eight XCDs in turn, each with an L2 of its own (4 MB).  An XCD takes every eighth tile of
    // base points and walks, for one block of hq query tiles after the other, through all its base tiles: the
    // workgroups in flight on it share those hq query tiles (hq x 213 KB at dim 200) and a handful of base tiles,
    // so both operands come from that L2 and each base tile from memory once per block of queries.
    // grid.x = 8 x ceil(base tiles / 8) x query blocks x hq.
    const int nqt = (nq + MT - 1) / MT;
    const unsigned xcd = blockIdx.x & 7u, place = blockIdx.x >> 3;
    const unsigned nbt8 = (unsigned)((ntiles + 7) >> 3);
    const unsigned qb = place / (nbt8 * (unsigned)hq), rem = place - qb * nbt8 * (unsigned)hq;
    const int64_t bt = (int64_t)(rem / (unsigned)hq) * 8 + xcd;
    const int qt = (int)(qb * (unsigned)hq + rem % (unsigned)hq);
    const int64_t b0 = (tile_step > 0 ? bt * tile_step : bt + bt / (-tile_step - 1) + 1) * NT;
    const int q0 = qt * MT;
    if (bt >= ntiles || b0 >= nb || qt >= nqt) return;  // padding: the last group of eight base tiles, the last query block
    constexpr int KS = kStageDims<NP>, NB = NP == 1 ? 4 : 2;
    const int stages = (dim + KS - 1) / KS;
    // staging: thread t copies 4 x 16 bytes of the query stage and splits row t/2, dimensions (t&1)*8 .. +8 (of either
    // half of the stage) of the base; rows beyond the end read the last row instead: their results are never written
    const int lrow = tid >> 1, lk = (tid & 1) * 8;
    const _Float16* pa = queries + (size_t)qt * stages * kStageA + tid * 8;
    const int64_t brow = min(b0 + lrow, nb - 1);
    const float* pb = base + (size_t)brow * dim + lk;
    const float bscale = mf_pow2(mf_scale_exp(bn[brow]));
    // A stage's loads are requested two stages ahead, with no condition, so that the wait for one stage's leaves the
    // next one's in flight (against one stage ahead: 10 000 x 1 000 000 x 200 in 18.4 instead of 19.1 ms).
    struct Staged {
        v8h a[4];
        float4 b[NB];
    } r0, r1;
    auto fetch = [&](int st, Staged& r) {
        st = min(st, stages - 1);
#pragma unroll
        for (int u = 0; u < 4; ++u) r.a[u] = *reinterpret_cast<const v8h*>(pa + (size_t)st * kStageA + u * 2048);
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int d = st * KS + (u >> 1) * BK + 4 * (u & 1);  // beyond dim (a multiple of 4) the row's start is read and then dropped
            r.b[u] = *reinterpret_cast<const float4*>(pb + (d + lk < dim ? d : -lk));
        }
    };
    auto park = [&](int st, int buf, const Staged& r) {
#pragma unroll
        for (int u = 0; u < 4; ++u) *reinterpret_cast<v8h*>(&sa[buf][u * 2048 + tid * 8]) = r.a[u];
        float4 b[NB];
#pragma unroll
        for (int u = 0; u < NB; ++u) b[u] = r.b[u];
        if ((st + 1) * KS > dim) {
#pragma unroll
            for (int u = 0; u < NB; ++u)
                if (st * KS + (u >> 1) * BK + 4 * (u & 1) + lk >= dim) b[u] = make_float4(0, 0, 0, 0);
        }
        v8h hi, lo;
        mf_split8(b[0], b[1], bscale, hi, lo);
        *reinterpret_cast<v8h*>(&sb[buf][lrow * BK + lk]) = hi;
        if constexpr (NP == 1) mf_split8(b[2], b[3], bscale, lo, hi);  // (the plane behind it: the hi halves of 16 dimensions more)
        *reinterpret_cast<v8h*>(&sb[buf][NT * BK + lrow * BK + lk]) = lo;
    };
    v16f acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
    const int kh = lane >> 5, m = lane & 31;  // an MFMA operand: lane = row (or column) m, dimensions kh * 8 .. + 7
    auto multiply = [&](int buf, int st) {
        const _Float16* A = &sa[buf][(wr * 128 + m) * BK + kh * 8];
        const _Float16* B = &sb[buf][(wc * 64 + m) * BK + kh * 8];
        v8h ah[4], al[4], bh[2], bl[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) bh[j] = *reinterpret_cast<const v8h*>(B + j * 32 * BK);
#pragma unroll
        for (int i = 0; i < 4; ++i) ah[i] = *reinterpret_cast<const v8h*>(A + i * 32 * BK);
#pragma unroll
        for (int j = 0; j < 2; ++j) bl[j] = *reinterpret_cast<const v8h*>(B + NT * BK + j * 32 * BK);
#pragma unroll
        for (int i = 0; i < 4; ++i) al[i] = *reinterpret_cast<const v8h*>(A + MT * BK + i * 32 * BK);
        auto product = [&](const v8h (&x)[4], const v8h (&y)[2]) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if constexpr (MODE == kLevels)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(y[j], x[i], acc[i][j], 0, 0, 0);
                    else
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[i], y[j], acc[i][j], 0, 0, 0);
                }
        };
        product(ah, bh);
        if constexpr (NP == 1) {
            if (st * KS + BK < dim) product(al, bl);  // (the last stage may hold 16 dimensions or fewer)
        } else {
            product(ah, bl);
            product(al, bh);
        }
    };
    fetch(0, r0);
    fetch(1, r1);
    park(0, 0, r0);
    __syncthreads();
#pragma unroll 1
    for (int st = 0; st + 1 < stages; st += 2) {
        fetch(st + 2, r0);
        multiply(0, st);
        park(st + 1, 1, r1);
        __syncthreads();
        fetch(st + 3, r1);
        multiply(1, st + 1);
        park(min(st + 2, stages - 1), 0, r0);
        __syncthreads();
    }
    if (stages & 1) multiply(0, stages - 1);
    __syncthreads();
    if constexpr (MODE == kLevels) {
        constexpr int kPitch = NT / 2 + 4;  // bytes of a query's levels in LDS, one bank on from query to query
        float* scol = reinterpret_cast<float*>(&sb[0][0]);  // what a base point contributes: its inverse scale, |b|^2
        float* sn2 = scol + NT;
        unsigned char* slev = reinterpret_cast<unsigned char*>(&sa[0][0]);
        static_assert(MT * kPitch <= (int)sizeof(sa) && 2 * NT * 4 <= (int)sizeof(sb), "the levels of a tile fit the operand buffers");
        if (tid < NT) {
            const int64_t c = b0 + tid;
            const float n2 = c < nb ? bn[c] : 0.0f;
            const bool takes_part = n2 <= 1.0e37f;
            scol[tid] = takes_part ? mf_pow2(-mf_scale_exp(n2)) : 0.0f;
            sn2[tid] = takes_part ? (L2 ? n2 : 0.0f) : -3.0e38f;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int rl = wr * 128 + i * 32 + m, r = q0 + rl;
            const float n2 = r < nq ? qn[r] : 0.0f;
            const float4 range = r < nq ? ranges[r] : make_float4(0, 0, 0, 0);  // origin, 1 / step (0: everything is level 0)
            const float inv = range.y;
            const float scale = (L2 ? -2.0f : -1.0f) * mf_pow2(-mf_scale_exp(n2)) * inv, off = ((L2 ? n2 : 0.0f) - range.x) * inv;
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int cl = wc * 64 + j * 32 + 8 * g + 4 * kh;
                    const float4 c4 = *reinterpret_cast<const float4*>(scol + cl), n4 = *reinterpret_cast<const float4*>(sn2 + cl);
                    const float cs[4] = {c4.x, c4.y, c4.z, c4.w}, cn[4] = {n4.x, n4.y, n4.z, n4.w};
                    uint32_t four = 0;
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        // (a value below the origin, or NaN, converts to 0)
                        const float u = __fmaf_rn(acc[i][j][4 * g + w] * cs[w], scale, __fmaf_rn(cn[w], inv, off));
                        four |= (uint32_t)fminf(fmaxf(u, 0.0f), 14.0f) << (4 * w);
                    }
                    *reinterpret_cast<uint16_t*>(slev + rl * kPitch + (cl >> 1)) = (uint16_t)four;
                }
        }
        __syncthreads();
        for (int i = tid; i < MT * 4; i += 256) {
            const int rl = i >> 2, piece = i & 3;
            if (q0 + rl >= nq) continue;
            const uint32_t* src = reinterpret_cast<const uint32_t*>(slev + rl * kPitch + piece * 16);
            *reinterpret_cast<uint4*>(levels + (size_t)(q0 + rl) * pitch + (size_t)(b0 >> 1) + piece * 16) =
                make_uint4(src[0], src[1], src[2], src[3]);
        }
        return;
    }
    // a 32 x 32 block's 16 registers: register v of lane l holds row 8 (v / 4) + 4 (l / 32) + v % 4, column l % 32.
    // What the tile's rows and columns contribute comes through LDS, fetched once per workgroup instead of by
    // dependent global loads per lane: norm and inverse scale of every row and column (times -2 or -1), the bounds.
    float* srow = reinterpret_cast<float*>(&sa[0][0]);  // the operand buffers are free after the last barrier of the loop
    float* srsc = srow + MT;
    float* stau = srsc + MT;
    float* scol = stau + MT;
    float* scsc = scol + NT;
    float* spre = scsc + NT + 4;
    unsigned int& s_nhit = *reinterpret_cast<unsigned int*>(scsc + NT);
    // (FUSED) the tile's entries that pass: ord(value) << 32 | row << 8 | column
    unsigned long long* shit = reinterpret_cast<unsigned long long*>(&sb[0][0]);
    constexpr int kHitCap = 2 * kStageB * 2 / 8;
    const float inf = __int_as_float(0x7f800000), nan = __int_as_float(0x7fc00000);
    {
        const int r = q0 + tid;
        const float n2 = r < nq ? qn[r] : 0.0f;
        srow[tid] = L2 ? n2 : 0.0f;
        srsc[tid] = mf_pow2(-mf_scale_exp(n2));
        if constexpr (FUSED) {
            const float t = r < nq ? tau[r] : -inf;
            stau[tid] = t;
            // What acc rs csc + |b|^2 cannot exceed where the value below does not exceed t.  Either sum is within
            // 2^-24 (2 |q|^2 + 3 |b|^2 + 2 t) of itself, and |b|^2 <= 2 (|q|^2 + t) wherever the value is at most t (the
            // inner product's two are the same sum).
            spre[tid] = L2 ? (t - n2) + 1.0e-6f * (n2 + fabsf(t)) : t;
        }
    }
    if (tid < NT) {
        // what a column adds to its entries: |b|^2 (L2) or 0, +inf for a tombstoned id; (FUSED) NaN beyond the end of
        // the base, which no comparison passes
        const int64_t c = b0 + tid;
        float v = FUSED ? nan : 0.0f, n2 = 0.0f;
        if (c < nb) {
            n2 = bn[c];
            v = L2 ? n2 : 0.0f;
            if (deleted) {
                const int64_t id = base_id0 + c;
                if ((deleted[id >> 5] >> (id & 31)) & 1u) v = inf;
            }
        }
        scol[tid] = v;
        scsc[tid] = (L2 ? -2.0f : -1.0f) * mf_pow2(-mf_scale_exp(n2));
    }
    if (tid == 0) s_nhit = 0u;
    __syncthreads();
    auto emit = [&](int rl, int cl, uint32_t ov) {
        const int r = q0 + rl;
        const unsigned pos = atomicAdd(&cnt[(size_t)r * kCntStride], 1u);
        if (pos < (unsigned)cap) lists[(size_t)r * cap + pos] = ((unsigned long long)ov << 32) | (uint32_t)(base_id0 + b0 + cl);
    };
#pragma unroll
    for (int ti = 0; ti < 4; ++ti) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {  // the 16 rows this lane holds of a block: four runs of four
            const int rl0 = wr * 128 + ti * 32 + 8 * g + 4 * kh;
            const float4 rn4 = *reinterpret_cast<const float4*>(srow + rl0);
            const float4 rs4 = *reinterpret_cast<const float4*>(srsc + rl0);
            float4 tq4 = make_float4(0, 0, 0, 0), pre4 = tq4;
            if constexpr (FUSED) tq4 = *reinterpret_cast<const float4*>(stau + rl0), pre4 = *reinterpret_cast<const float4*>(spre + rl0);
            const float rn[4] = {rn4.x, rn4.y, rn4.z, rn4.w}, rs[4] = {rs4.x, rs4.y, rs4.z, rs4.w};
            const float tq[4] = {tq4.x, tq4.y, tq4.z, tq4.w}, pre[4] = {pre4.x, pre4.y, pre4.z, pre4.w};
#pragma unroll
            for (int tj = 0; tj < 2; ++tj) {
                const int cl = wc * 64 + tj * 32 + m;
                const float bnc = scol[cl], csc = scsc[cl];
                if constexpr (FUSED && NP == 1) {
                    // (most fours hold nothing that passes: three instructions an entry and one branch for the four; 3 % of
                    // the call on one product, nothing on three, which smaller batches with looser bounds take)
                    bool any = false;
#pragma unroll
                    for (int w = 0; w < 4; ++w) any |= __fmaf_rn(acc[ti][tj][4 * g + w], rs[w] * csc, bnc) <= pre[w];
                    if (__ballot(any) == 0ull) continue;
                }
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    // (|q|^2 + |b|^2) - 2 q.b, or -q.b; a tombstoned column's +inf survives both forms
                    const float sv = __fmaf_rn(acc[ti][tj][4 * g + w], rs[w] * csc, L2 ? rn[w] + bnc : bnc);
                    if constexpr (FUSED) {
                        if (sv <= tq[w]) {  // rows beyond nq have tau = -inf, columns beyond nb give NaN
                            const unsigned pos = atomicAdd(&s_nhit, 1u);
                            if (pos < (unsigned)kHitCap)
                                shit[pos] = ((unsigned long long)mf_ord32(sv) << 32) | (unsigned)((rl0 + w) << 8) | (unsigned)cl;
                            else  // more hits than the tile's buffer holds: straight to the list
                                emit(rl0 + w, cl, mf_ord32(sv));
                        }
                    } else {
                        const int r = q0 + rl0 + w;
                        if (r < nq && b0 + cl < nb) D[(size_t)r * ldD + bt * NT + cl] = sv;
                    }
                }
            }
        }
    }
    if constexpr (FUSED) {
        __syncthreads();
        const int nhit = (int)min(s_nhit, (unsigned)kHitCap);
        for (int i = tid; i < nhit; i += 256) {
            const unsigned long long h = shit[i];
            emit((int)((h >> 8) & 0xffu), (int)(h & 0xffu), (uint32_t)(h >> 32));
        }
    }
}

// What one product of hi halves (NP = 1) is off by beside the accumulation: |q.b - hi(q).hi(b)| <= |q - hi(q)| |b| +
// |hi(q)| |b - hi(b)|, for any row of the index.
__device__ __forceinline__ float mf_hi_loss(float qn, float qres, const uint32_t* bn_max_bits, const uint32_t* bres_max_bits) {
    const float bmax = sqrtf(__uint_as_float(*bn_max_bits)), bres = __uint_as_float(*bres_max_bits);
    return (qres * bmax + (sqrtf(qn) + qres) * bres) * (1.0f + 1.0e-4f);
}

// The range of a query's levels from the distances to a sample of the base (one wavefront per query): fourteen steps from
// 3.5 standard deviations below the mean to 0.1 above, where a search's thresholds fall from its first round to its last.
// ranges[q]: origin, 1 / step, step, and the bound E on |the tile kernel's value of an entry - its exact distance|:
// what one product loses (mf_hi_loss); (7 dim + 32) u n2 for the accumulation, the norms and the final additions (head of
// this file) and (dim + 8) u d for the reference order, d <= 2 n2; and what the value that is cut into steps is off by,
// the roundings of its sums of |q|^2, |b|^2, 2 |q| |b| and the origin and of 1 / step, 32 u (n2 + |origin|).  A query or a sample that is
// not finite gets 1 / step = 0: level 0 everywhere, which says nothing.
// unfit (or null): *unfit += 1 where the levels would settle little: E is more than two and a quarter steps, or half of the
// sample lies within two widened steps of its smallest entry (one huge row in the sample, and a step is wider than the
// others' whole spread).  The line: the time of a search with levels over the time without, 60 000 .. 80 000 rows of 132 ..
// 1028 floats with an offset common to all or one row times 3 .. 1000, L = 128 .. 400.  With E of 0.02 .. 2.2 steps, as data
// without either and up to an offset of five standard deviations (512 floats) have it, 0.30 .. 0.92; 2.7 .. 3.7 steps 0.87 ..
// 1.27; 6 .. 10 0.87 .. 1.94; beyond, one row times 30 and more, 1.26 .. 2.2.  Half of the sample: 0.83 and more of it lay further out
// where a row in it was three times as long (0.82 .. 0.99), 0.03 and less where it was ten times as long (1.13 .. 2.1).
__global__ __launch_bounds__(64) void level_ranges_kernel(const float* __restrict__ D, int64_t ldD, int n, int dim, int metric,
                                                         const float* __restrict__ qn, const uint32_t* __restrict__ bn_max_bits,
                                                         const float* __restrict__ qres, const uint32_t* __restrict__ bres_max_bits,
                                                         float4* __restrict__ ranges, int* __restrict__ unfit) {
    const int q = blockIdx.x, lane = threadIdx.x;
    const float* row = D + (size_t)q * ldD;
    float sum = 0.0f;
    for (int i = lane; i < n; i += 64) sum += row[i];
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    const float mean = sum / (float)n;
    float var = 0.0f;
    for (int i = lane; i < n; i += 64) var = __fmaf_rn(row[i] - mean, row[i] - mean, var);
    for (int off = 32; off > 0; off >>= 1) var += __shfl_xor(var, off, 64);
    const float sd = sqrtf(var / (float)n), origin = mean - 3.5f * sd, step = sd * (3.6f / 14.0f), inv = 1.0f / step;
    const float n2 = qn[q] + fminf(__uint_as_float(*bn_max_bits), 1.0e37f);  // (larger rows take no part)
    const float u = 5.9604645e-8f;
    const float E = (metric == 0 ? 2.0f : 1.0f) * mf_hi_loss(qn[q], qres[q], bn_max_bits, bres_max_bits) +
                    (float)(9 * dim + 64) * u * n2 + 32.0f * u * (n2 + fabsf(origin)) + 1.0e-30f;
    const bool good = n2 <= 1.0e38f && E <= 1.0e38f && inv <= 1.0e20f && inv >= 1.0e-15f && fabsf(origin) <= 1.0e38f;
    if (lane == 0) ranges[q] = good ? make_float4(origin, inv, step, E) : make_float4(0, 0, 0, 0);
    if (!unfit) return;
    float least = 3.402823466e+38f;
    for (int i = lane; i < n; i += 64) least = fminf(least, row[i]);
    for (int off = 32; off > 0; off >>= 1) least = fminf(least, __shfl_xor(least, off, 64));
    int beyond = 0;
    for (int i = lane; i < n; i += 64) beyond += row[i] - least > 2.0f * (step + 2.0f * E);
    for (int off = 32; off > 0; off >>= 1) beyond += __shfl_xor(beyond, off, 64);
    if (lane == 0 && !(good && E <= 2.25f * step && 2 * beyond >= n)) atomicAdd(unfit, 1);
}

// How many entries of a sample of the base lie so close behind the bound that NP = 1 could not tell them from the
// entries before it: one workgroup per query counts those up to tau + 2 loss; *extra += count - kc.
__global__ __launch_bounds__(256) void count_close_kernel(const float* __restrict__ D, int64_t ldD, int64_t n, int kc, int metric,
                                                        const float* __restrict__ qn, const uint32_t* __restrict__ bn_max_bits,
                                                        const float* __restrict__ qres, const uint32_t* __restrict__ bres_max_bits,
                                                        const float* __restrict__ tau, int* __restrict__ extra) {
    const int q = blockIdx.x;
    const float loss = (metric == 0 ? 2.0f : 1.0f) * mf_hi_loss(qn[q], qres[q], bn_max_bits, bres_max_bits);
    const float upto = tau[q] + 2.0f * loss;
    int c = 0;
    __shared__ int s_count;
    if (threadIdx.x == 0) s_count = 0;
    __syncthreads();
    for (int64_t i = threadIdx.x; i < n; i += 256) c += D[(size_t)q * ldD + i] <= upto;
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
    if ((threadIdx.x & 63) == 0) atomicAdd(&s_count, c);
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(extra, max(0, s_count - kc));
}

__device__ __forceinline__ float rerank_add(const float4 a, const float4 b, float s, int metric) {
    if (metric == 0) {
        float t;
        t = a.x - b.x, s = __fmaf_rn(t, t, s);
        t = a.y - b.y, s = __fmaf_rn(t, t, s);
        t = a.z - b.z, s = __fmaf_rn(t, t, s);
        t = a.w - b.w, s = __fmaf_rn(t, t, s);
    } else {
        s = __fmaf_rn(a.x, b.x, s), s = __fmaf_rn(a.y, b.y, s), s = __fmaf_rn(a.z, b.z, s), s = __fmaf_rn(a.w, b.w, s);
    }
    return s;
}

// One workgroup per query: the kc candidates (ids, -1 = none; approximate signed distances, ascending) are measured
// in the reference's order (one thread walks the dimensions of one candidate with one fused multiply-add each,
// include/utils.cuh:254-275, 307-323: the arithmetic of distance_tile_kernel), sorted by (distance, id), and the k
// best written.  redo[q] = 1 when the result cannot be vouched for (see the head of this file); redo[number of queries] =
// *lost: the call reads both after one wait.
__global__ __launch_bounds__(256) void rerank_kernel(const float* __restrict__ queries, const float* __restrict__ base,
                                                    int dim, int metric, const int32_t* __restrict__ cand_ids,
                                                    const float* __restrict__ cand_d, int kc, int k,
                                                    const float* __restrict__ qn, const uint32_t* __restrict__ bn_max_bits,
                                                    const float* __restrict__ qres, const uint32_t* __restrict__ bres_max_bits,
                                                    int32_t* __restrict__ ids, float* __restrict__ dists,
                                                    int* __restrict__ redo, const int* __restrict__ lost) {
    extern __shared__ unsigned long long rkeys[];
    const int q = blockIdx.x, tid = threadIdx.x;
    int P = 2;
    while (P < kc) P <<= 1;
    const float* qv = queries + (size_t)q * dim;
    for (int i = tid; i < P; i += 256) {
        unsigned long long key = ~0ull;
        const int32_t id = i < kc ? cand_ids[(size_t)q * kc + i] : -1;
        if (id >= 0) {
            const float4* b4 = reinterpret_cast<const float4*>(base + (size_t)id * dim);
            const float4* q4 = reinterpret_cast<const float4*>(qv);
            float s = 0.0f;
            // eight loads of the row on their way at a time: few threads have a row, and each waits for its own
            int c = 0;
            for (; c + 8 <= dim / 4; c += 8) {
                float4 b[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) b[u] = b4[c + u];
#pragma unroll
                for (int u = 0; u < 8; ++u) s = rerank_add(q4[c + u], b[u], s, metric);
            }
            for (; c < dim / 4; ++c) s = rerank_add(q4[c], b4[c], s, metric);
            if (metric != 0) s = 0.0f - s;
            key = ((unsigned long long)mf_ord32(s) << 32) | (uint32_t)id;
        }
        rkeys[i] = key;
    }
    __syncthreads();
    for (int k2 = 2; k2 <= P; k2 <<= 1)
        for (int j = k2 >> 1; j > 0; j >>= 1) {
            for (int t = tid; t < (P >> 1); t += 256) {
                const int i = 2 * t - (t & (j - 1)), x = i + j;
                const bool asc = (i & k2) == 0;
                const unsigned long long ka = rkeys[i], kb = rkeys[x];
                if ((ka > kb) == asc) rkeys[i] = kb, rkeys[x] = ka;
            }
            __syncthreads();
        }
    for (int i = tid; i < k; i += 256) {
        const unsigned long long key = rkeys[i];
        const bool none = key == ~0ull;
        ids[(size_t)q * k + i] = none ? -1 : (int32_t)(uint32_t)key;
        if (dists) {
            const float s = mf_unord32((uint32_t)(key >> 32));
            const float far = 3.402823466e+38f;
            dists[(size_t)q * k + i] = none ? (metric == 0 ? far : -far) : (metric == 0 ? s : 0.0f - s);
        }
    }
    if (tid == 0) {
        // Where |q|^2 + |b|^2 is infinite or NaN, or twice it is, approximate distances may be so too: such points were
        // dropped like tombstoned ones, and a list that is not full says nothing.
        const float n2 = qn[q] + __uint_as_float(*bn_max_bits);
        int bad = !(n2 <= 1.5e38f);
        // otherwise every live point is a candidate unless the list is full; a full list vouches for the k best only if
        // the k-th of them lies clear of the worst candidate's approximate distance
        if (!bad && cand_ids[(size_t)q * kc + kc - 1] >= 0) {
            const float worst = cand_d[(size_t)q * kc + kc - 1];
            const float u = 5.9604645e-8f, un2 = u * n2;
            const float delta = (metric == 0 ? (float)(7 * dim + 32) * un2 + (float)(dim + 8) * (u * fmaxf(worst, 0.0f))
                                             : (float)(4 * dim + 32) * un2) +
                                (float)(10 * dim + 40) * 1.4e-45f +
                                (qres ? (metric == 0 ? 2.0f : 1.0f) * mf_hi_loss(qn[q], qres[q], bn_max_bits, bres_max_bits) : 0.0f);
            const unsigned long long kth = rkeys[k - 1];
            const float sk = mf_unord32((uint32_t)(kth >> 32));
            if (kth == ~0ull || !(sk < worst - delta)) bad = 1;
        }
        redo[q] = bad;
        if (q == 0) redo[gridDim.x] = lost ? *lost : 0;
    }
}

// dst[rows[i]][0..k) = src[i][0..k)
__global__ void scatter_results_kernel(const int32_t* __restrict__ rows, int count, int k, const int32_t* __restrict__ src_ids,
                                       const float* __restrict__ src_d, int32_t* __restrict__ dst_ids,
                                       float* __restrict__ dst_d) {
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < (int64_t)count * k;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(t / k), j = (int)(t - (int64_t)i * k);
        dst_ids[(size_t)rows[i] * k + j] = src_ids[t];
        if (dst_d) dst_d[(size_t)rows[i] * k + j] = src_d[t];
    }
}

}  // namespace

hipError_t launch_row_norms(const float* x, int64_t n, int dim, float* out, uint32_t* max_bits, uint32_t* res_max,
                            hipStream_t stream) {
    if (n <= 0) return hipErrorInvalidValue;
    const int64_t blocks = std::min<int64_t>((n + 3) / 4, 2048);  // 32 wavefronts per compute unit
    hipLaunchKernelGGL(row_norms_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, x, n, dim, out, max_bits, res_max);
    return hipGetLastError();
}

namespace {
int stages_of(int dim, int products) { return products == 1 ? (dim + kStageDims<1> - 1) / kStageDims<1> : (dim + BK - 1) / BK; }
}  // namespace

size_t split_queries_bytes(int nq, int dim, int products) {
    return (size_t)((nq + MT - 1) / MT) * stages_of(dim, products) * kStageA * sizeof(_Float16);
}

size_t split_queries_offset(int64_t row, int dim, int products) {
    return (size_t)(row / MT) * stages_of(dim, products) * kStageA * sizeof(_Float16);
}

hipError_t launch_prepare_queries(const float* queries, int nq, int dim, int products, float* qn, float* res, void* out,
                                  unsigned int* cnt, int* zero, hipStream_t stream) {
    const int tiles = (nq + MT - 1) / MT;
    if (nq <= 0) return hipErrorInvalidValue;
    auto kernel = products == 1 ? prepare_queries_kernel<1> : prepare_queries_kernel<3>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)tiles * (MT / 4)), dim3(256), 0, stream, queries, nq, dim, stages_of(dim, products),
                       qn, res, static_cast<_Float16*>(out), cnt, zero);
    return hipGetLastError();
}

namespace {
// the launch geometry: query tiles an XCD keeps in its L2 while it walks the base (about 2 MB of them), and the grid
bool tile_grid(int nq, int dim, int products, int64_t ntiles, int64_t* hq, unsigned* wgs) {
    const int64_t nqt = (nq + MT - 1) / MT;
    const int64_t per_tile = (int64_t)stages_of(dim, products) * kStageA * (int64_t)sizeof(_Float16);
    const int64_t want = std::max<int64_t>(1, ((int64_t)2 << 20) / per_tile);
    const int64_t qblocks = (nqt + want - 1) / want;
    *hq = (nqt + qblocks - 1) / qblocks;
    const int64_t total = (ntiles + 7) / 8 * 8 * qblocks * *hq;
    *wgs = (unsigned)total;
    return nq > 0 && ntiles > 0 && total <= 0x7fffffff;
}
}  // namespace

hipError_t launch_approx_tile(const void* queries, const float* base, int nq, int64_t nb, int dim, int metric, int products,
                              const float* qn, const float* bn, const uint32_t* deleted, int64_t base_id0, float* D,
                              int64_t ldD, hipStream_t stream, int64_t sample_tiles, int tile_stride) {
    const int64_t ntiles = sample_tiles > 0 ? sample_tiles : (nb + NT - 1) / NT;
    int64_t hq = 0;
    unsigned wgs = 0;
    if (!tile_grid(nq, dim, products, ntiles, &hq, &wgs) || tile_stride < 1) return hipErrorInvalidValue;
    auto kernel = products == 1 ? (metric == 0 ? approx_tile_mfma_kernel<kMatrix, true, 1> : approx_tile_mfma_kernel<kMatrix, false, 1>)
                                : (metric == 0 ? approx_tile_mfma_kernel<kMatrix, true, 3> : approx_tile_mfma_kernel<kMatrix, false, 3>);
    hipLaunchKernelGGL(kernel, dim3(wgs), dim3(256), 0, stream, static_cast<const _Float16*>(queries), base, nq, nb, dim, qn,
                       bn, deleted, base_id0, ntiles, tile_stride, (int)hq, D, ldD, (const float*)nullptr,
                       (unsigned long long*)nullptr, (int64_t)0, (unsigned int*)nullptr, (const float4*)nullptr,
                       (unsigned char*)nullptr, (size_t)0);
    return hipGetLastError();
}

hipError_t launch_approx_filter(const void* queries, const float* base, int nq, int64_t nb, int dim, int metric, int products,
                                const float* qn, const float* bn, const uint32_t* deleted, const float* tau,
                                unsigned long long* lists, int64_t cap, unsigned int* cnt, int tile_step,
                                hipStream_t stream) {
    const int64_t all = (nb + NT - 1) / NT;
    const int64_t step = tile_step < 0 ? -(int64_t)tile_step : tile_step;
    if (tile_step == 0 || tile_step == -1 || nb > 0x7fffffff) return hipErrorInvalidValue;
    const int64_t multiples = (all + step - 1) / step, ntiles = tile_step > 0 ? multiples : all - multiples;
    if (ntiles == 0) return hipSuccess;  // no tile between the multiples
    int64_t hq = 0;
    unsigned wgs = 0;
    if (!tile_grid(nq, dim, products, ntiles, &hq, &wgs)) return hipErrorInvalidValue;
    auto kernel = products == 1 ? (metric == 0 ? approx_tile_mfma_kernel<kFused, true, 1> : approx_tile_mfma_kernel<kFused, false, 1>)
                                : (metric == 0 ? approx_tile_mfma_kernel<kFused, true, 3> : approx_tile_mfma_kernel<kFused, false, 3>);
    hipLaunchKernelGGL(kernel, dim3(wgs), dim3(256), 0, stream, static_cast<const _Float16*>(queries), base, nq, nb, dim, qn,
                       bn, deleted, (int64_t)0, ntiles, tile_step, (int)hq, (float*)nullptr, (int64_t)0, tau, lists, cap, cnt,
                       (const float4*)nullptr, (unsigned char*)nullptr, (size_t)0);
    return hipGetLastError();
}

hipError_t launch_level_ranges(const float* D, int64_t ldD, int nq, int n, int dim, int metric, const float* qn,
                               const uint32_t* bn_max_bits, const float* qres, const uint32_t* bres_max_bits, float4* ranges,
                               int* unfit, hipStream_t stream) {
    hipLaunchKernelGGL(level_ranges_kernel, dim3(nq), dim3(64), 0, stream, D, ldD, n, dim, metric, qn, bn_max_bits, qres,
                       bres_max_bits, ranges, unfit);
    return hipGetLastError();
}

size_t level_pitch(int64_t n) { return (size_t)((n + NT - 1) / NT) * (NT / 2); }

hipError_t launch_levels(const void* queries, const float* base, int nq, int64_t nb, int dim, int metric, const float* qn,
                         const float* bn, const float4* ranges, unsigned char* levels, hipStream_t stream) {
    const int64_t ntiles = (nb + NT - 1) / NT;
    int64_t hq = 0;
    unsigned wgs = 0;
    if (!tile_grid(nq, dim, 1, ntiles, &hq, &wgs)) return hipErrorInvalidValue;
    auto kernel = metric == 0 ? approx_tile_mfma_kernel<kLevels, true, 1> : approx_tile_mfma_kernel<kLevels, false, 1>;
    hipLaunchKernelGGL(kernel, dim3(wgs), dim3(256), 0, stream, static_cast<const _Float16*>(queries), base, nq, nb, dim, qn,
                       bn, (const uint32_t*)nullptr, (int64_t)0, ntiles, 1, (int)hq, (float*)nullptr, (int64_t)0,
                       (const float*)nullptr, (unsigned long long*)nullptr, (int64_t)0, (unsigned int*)nullptr, ranges, levels,
                       level_pitch(nb));
    return hipGetLastError();
}

hipError_t launch_rerank(const float* queries, const float* base, int nq, int dim, int metric, const int32_t* cand_ids,
                         const float* cand_d, int kc, int k, const float* qn, const uint32_t* bn_max_bits, const float* qres,
                         const uint32_t* bres_max_bits, int32_t* ids, float* dists, int* redo, const int* lost,
                         hipStream_t stream) {
    int P = 2;
    while (P < kc) P <<= 1;
    hipLaunchKernelGGL(rerank_kernel, dim3(nq), dim3(256), (size_t)P * 8, stream, queries, base, dim, metric, cand_ids,
                       cand_d, kc, k, qn, bn_max_bits, qres, bres_max_bits, ids, dists, redo, lost);
    return hipGetLastError();
}

hipError_t launch_count_close(const float* D, int64_t ldD, int nq, int64_t n, int kc, int metric, const float* qn,
                              const uint32_t* bn_max_bits, const float* qres, const uint32_t* bres_max_bits, const float* tau,
                              int* extra, hipStream_t stream) {
    hipLaunchKernelGGL(count_close_kernel, dim3(nq), dim3(256), 0, stream, D, ldD, n, kc, metric, qn, bn_max_bits, qres,
                       bres_max_bits, tau, extra);
    return hipGetLastError();
}

hipError_t launch_scatter_results(const int32_t* rows, int count, int k, const int32_t* src_ids, const float* src_d,
                                  int32_t* dst_ids, float* dst_d, hipStream_t stream) {
    int64_t blocks = ((int64_t)count * k + 255) / 256;
    blocks = blocks > 4096 ? 4096 : (blocks < 1 ? 1 : blocks);
    hipLaunchKernelGGL(scatter_results_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, rows, count, k, src_ids, src_d,
                       dst_ids, dst_d);
    return hipGetLastError();
}

}  // namespace coral
