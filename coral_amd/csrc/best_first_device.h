// best_first_device.h -- the best-first kernel with the beam in registers (device code; instantiated for one wavefront
// per query in best_first.hip and for four in best_first_shared.hip).  What it does and why: best_first.hip.
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "beam_search.h"
#include "search_device.h"

namespace coral {

namespace {

constexpr int kWavesPerWg = 4;
constexpr int kNoPlace = 0x7fffffff;
constexpr int kBatch = 32;  // ids measured and merged at a time (a graph row has at most 32)
constexpr int kScreenRows = 8;  // half-precision rows in flight per group of 32 lanes in the screening phase

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The beam.  L keys in ascending order, spread over the wavefront's registers: KPL consecutive keys per lane, the
// last one in the last register of lane 63 (capacity C = 64 KPL >= L; the C - L places in front hold kFront, smaller
// than any key and flagged as expanded).  Places not filled yet hold kKeyMax, which is flagged as well.  So the worst
// entry of a full beam is always the same register of the same lane, and a key that is inserted pushes exactly the
// last one out.
constexpr uint64_t kFront = 1ull;

// One key, the same in every lane: a place whose key is larger takes the larger of the new key and its left
// neighbour's.  Five instructions per place and one exchange with the lane below -- no search, no memory, no order in
// which the candidates of a step must come.  (In LDS, with ranks, binary searches and a byte counter per place, a
// step's four to five candidates took 3600 of a step's 16 000 cycles with sixteen wavefronts per CU at L = 512.)
template <int KPL>
__device__ __forceinline__ void beam_insert(uint64_t (&r)[KPL], uint64_t key) {
    const uint32_t plo = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)kFront, (int)(uint32_t)r[KPL - 1], 0x138, 0xF, 0xF, false);
    const uint32_t phi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(r[KPL - 1] >> 32), 0x138, 0xF, 0xF, false);  // wave_shr:1
    const uint64_t before = ((uint64_t)phi << 32) | plo;
    bool less = key < r[KPL - 1];
#pragma unroll
    for (int j = KPL - 1; j > 0; --j) {
        const bool left = key < r[j - 1];
        r[j] = less ? (left ? r[j - 1] : key) : r[j];
        less = left;
    }
    r[0] = less ? (key < before ? before : key) : r[0];
}

__device__ __forceinline__ uint64_t readlane_u64(uint64_t x, int lane) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), lane);
    return ((uint64_t)hi << 32) | lo;
}

// Distances of NU rows per group of G lanes: row u of group grp is entry first + u GPW + grp of the list, which holds
// valid ids up to its 32nd entry whatever T is.  The lane that files a row (rows_filed of them per group) gets its
// signed distance and its place in the list.  A wavefront-wide group reads its row through a scalar address; lanes past
// the row's end read its last chunk again and leave their sum as it was.
template <int G, int CPL, int NU>
__device__ __forceinline__ float measure_rows(const float* __restrict__ vec, const uint32_t* list, int first, int dim,
                                              int metric, const float4 (&q)[CPL], int& place) {
    constexpr int GPW = 64 / G;
    const int lane = threadIdx.x & 63, gl = lane & (G - 1), grp = lane / G, chunks = dim >> 2;
    float4 v[NU][CPL];
    if constexpr (G == 64) {
        const int ids = (int)list[lane & 31];
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int id = __builtin_amdgcn_readlane(ids, first + u);
            const float4* row = reinterpret_cast<const float4*>(vec + (uint64_t)(uint32_t)id * (uint32_t)dim);
#pragma unroll
            for (int t = 0; t < CPL; ++t) v[u][t] = row[min(gl + G * t, chunks - 1)];
        }
    } else {
        uint32_t id[NU];
#pragma unroll
        for (int u = 0; u < NU; ++u) id[u] = list[first + u * GPW + grp];
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const float4* row = reinterpret_cast<const float4*>(vec + (uint64_t)id[u] * (uint32_t)dim);
            v[u][0] = row[min(gl, chunks - 1)];
        }
    }
    float acc[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        float s = 0.0f;
#pragma unroll
        for (int t = 0; t < CPL; ++t) {
            const float before = s;
            if (metric == 0) {
                float d;
                d = q[t].x - v[u][t].x, s = __fmaf_rn(d, d, s);
                d = q[t].y - v[u][t].y, s = __fmaf_rn(d, d, s);
                d = q[t].z - v[u][t].z, s = __fmaf_rn(d, d, s);
                d = q[t].w - v[u][t].w, s = __fmaf_rn(d, d, s);
            } else {
                s = __fmaf_rn(q[t].x, v[u][t].x, s);
                s = __fmaf_rn(q[t].y, v[u][t].y, s);
                s = __fmaf_rn(q[t].z, v[u][t].z, s);
                s = __fmaf_rn(q[t].w, v[u][t].w, s);
            }
            s = gl + G * t < chunks ? s : before;
        }
        acc[u] = s;
    }
    const float sum = rows_sum<G, NU>(acc);
    place = gl < NU ? first + filed_row<G, NU>(lane) * GPW + grp : kNoPlace;
    return metric == 0 ? sum : 0.0f - sum;
}

// SCREEN: rows are first measured in a smaller copy of the vectors: 1 the half-precision copy (b.vec16; rows of more
// than 128 floats), 2 the copy in eight-bit codes (b.vec8; rows of 68 .. 512 floats).
// RIF: float4 registers of row data per lane that are requested before any is added up.  KPL: keys of the beam per lane.
// WGS: workgroups a CU is to hold, which sets the registers a lane may use.
// The visited state in HBM is a byte per node and slot, or (b.packed) one 32-bit word per 24 nodes, 8 bits of epoch
// over 24 flags: a sixth of the memory, the same one line per test.
// WPQ: wavefronts per query, 1 or 4.  Four share the rows of a step, for batches that leave a CU's other SIMDs idle
// and rows so wide that a step's would take a lone wavefront several passes: the first wavefront reads the graph row and
// tests the ids against the bitmap (the only form of the visited set here), each measures a quarter of the new ones, and
// each keeps a copy of the beam, to which all four add the same keys -- two barriers a step, and nothing else passes
// between them.  A workgroup then is one query, else four.
template <int G, int CPL, int RIF, int KPL, int SCREEN, int WGS, int WPQ>
__global__ __launch_bounds__(kWavesPerWg * 64, WGS) void best_first_wave_kernel(const SearchArgs a, const BestFirstArgs b) {
    static_assert(WPQ == 1 || WPQ == kWavesPerWg, "a workgroup is one query or one per wavefront");
    constexpr int kMine = kBatch / WPQ;  // rows of a step per wavefront
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int slot = WPQ > 1 ? (int)blockIdx.x : (int)blockIdx.x * b.waves_per_wg + wave;
    const int part = WPQ > 1 ? wave : 0;  // the wavefront's place among those of its query
    if (slot >= b.slots) return;  // the whole wavefront, and where a workgroup has barriers the whole workgroup
    const int L = a.L, R = a.R, dim = a.dim, chunks = dim >> 2, M = a.M;
    unsigned char* mine_lds = smem;
    if (WPQ == 1) mine_lds += (size_t)wave * best_first_wave_lds_bytes(b.bloom_log2, b.table_log2, b.coded_bytes, b.bitmap_words);
    // (WPQ > 1) the candidates of a step by their place in the list, the step's number of new ids (two, used in turn),
    // the query's number, the rows that the wavefronts read in fp32 and on
    // the smaller copy
    uint64_t* cand = reinterpret_cast<uint64_t*>(mine_lds);
    int* s_new = reinterpret_cast<int*>(cand + kBatch);
    int* s_qid = s_new + 2;
    int* s_exact = s_new + 3;
    int* s_screened = s_new + 4;
    uint32_t* lists = reinterpret_cast<uint32_t*>(mine_lds + (WPQ > 1 ? kSharedStepBytes - (WPQ - 1) * kBatch * 4 : 0));
    uint32_t* todo = lists;                                       // kBatch ids
    uint32_t* todo2 = lists + kBatch * (1 + part);                // kBatch ids: what the screening leaves to measure
    uint32_t* table = lists + kBatch * (1 + WPQ);                             // 2^table_log2 16-bit cells, or none (16-byte aligned)
    uint32_t* bits = table + (b.table_log2 ? (1 << b.table_log2) >> 1 : 0);  // a bitmap of all ids, or none
    uint32_t* bloom = bits + b.bitmap_words;                      // 2^bloom_log2 bits, or none
    const bool bitmap = b.bitmap_words != 0, packed = b.packed != 0;
    // The Bloom filter holds every id the query has visited.  An id it does not know is new for certain and needs no
    // look at the visited state in HBM (most tests: a query sees far more new ids than old ones); an id it may know
    // is looked up as before.  Two multiplicative hashes.
    const int bl = b.bloom_log2;
    const int bloom_words = bl ? (1 << bl) >> 5 : 0;
    signed char* qh8 = reinterpret_cast<signed char*>(bloom + bloom_words);  // the query in integer codes (SCREEN == 2)
    signed char* ql8 = qh8 + ((dim + 15) & ~15);
    auto bloom_bits = [&](uint32_t id, uint32_t& h1, uint32_t& h2) {
        h1 = (id * 0x9E3779B1u) >> (32 - bl);
        h2 = (id * 0x85EBCA77u + 0x3C6EF372u) >> (32 - bl);
    };
    auto bloom_may_hold = [&](uint32_t id) -> bool {
        uint32_t h1, h2;
        bloom_bits(id, h1, h2);
        return ((bloom[h1 >> 5] >> (h1 & 31)) & (bloom[h2 >> 5] >> (h2 & 31)) & 1u) != 0u;
    };
    auto bloom_add = [&](uint32_t id) {
        uint32_t h1, h2;
        bloom_bits(id, h1, h2);
        atomicOr(&bloom[h1 >> 5], 1u << (h1 & 31));
        atomicOr(&bloom[h2 >> 5], 1u << (h2 & 31));
    };

    // First level of the visited set, when the launch has one: an exact table of 16-bit cells in LDS, in buckets of
    // four.  A bijection mixes the id; the high bits of the result pick a bucket, a second bucket follows from that
    // one and the remaining bits (the remainder), and a cell stores the remainder and which of the two buckets it is
    // in: cell = 1 + ((second << rb) | remainder), 0 = empty.  (bucket, cell) determine the mixed value and hence the
    // id, so the table is exact.  A test reads the two buckets (two 8-byte reads, whatever the load); an id goes to
    // the emptier one.  0: the id was there; 1: it is now; 2: it is not and cannot be (both buckets are full): such
    // ids are settled against the state in HBM.
    // One call handles distinct ids in its lanes (the caller has removed repeats).
    const int tl = b.table_log2;
    const uint32_t t_bkmask = tl ? (1u << (tl - 2)) - 1u : 0u;
    const uint32_t t_bmask = b.id_bits >= 32 ? 0xffffffffu : (1u << b.id_bits) - 1u;
    const int t_rb = b.rem_bits, t_xs = b.id_bits > 1 ? b.id_bits / 2 : 1;
    const uint32_t t_rmask = (1u << t_rb) - 1u;
    auto table_test_and_set = [&](uint32_t id) -> int {
        uint32_t h = (id * 0x9E3779B1u) & t_bmask;
        h ^= h >> t_xs;
        h = (h * 0x85EBCA6Bu) & t_bmask;
        h ^= h >> t_xs;
        const uint32_t rem = h & t_rmask;
        const uint32_t b1 = (h >> t_rb) & t_bkmask;
        const uint32_t b2 = (b1 ^ (((rem + 1u) * 0x5BD1E995u) >> 15)) & t_bkmask;
        const uint32_t want1 = 1u + rem, want2 = 1u + ((1u << t_rb) | rem);
        const uint2* buckets = reinterpret_cast<const uint2*>(table);
        for (int attempt = 0; attempt < 8; ++attempt) {
            const uint2 w1 = buckets[b1], w2 = buckets[b2];
            const uint32_t c1[4] = {w1.x & 0xffffu, w1.x >> 16, w1.y & 0xffffu, w1.y >> 16};
            const uint32_t c2[4] = {w2.x & 0xffffu, w2.x >> 16, w2.y & 0xffffu, w2.y >> 16};
            int e1 = 0, e2 = 0, f1 = -1, f2 = -1;  // empty cells and the first of them, per bucket
            bool present = false;
#pragma unroll
            for (int i = 3; i >= 0; --i) {
                present |= c1[i] == want1 || c2[i] == want2;
                if (c1[i] == 0u) ++e1, f1 = i;
                if (c2[i] == 0u) ++e2, f2 = i;
            }
            if (present) return 0;
            if (e1 == 0 && e2 == 0) return 2;
            const bool second = e2 > e1;
            const uint32_t bk = second ? b2 : b1, want = second ? want2 : want1;
            const int cell = second ? f2 : f1;
            const uint32_t oldw = second ? (cell < 2 ? w2.x : w2.y) : (cell < 2 ? w1.x : w1.y);
            const int sh = (cell & 1) * 16;
            if (atomicCAS(table + bk * 2u + (uint32_t)(cell >> 1), oldw, oldw | (want << sh)) == oldw) return 1;
            // another lane took a cell of that word: look again
        }
        return 2;
    };

    uint8_t* vis = bitmap ? nullptr : b.visited + (size_t)slot * b.stride;
    uint32_t epoch = bitmap ? 0u : b.epochs[slot];

    constexpr int GPW = 64 / G;  // row groups per wavefront
    // rows in flight per group: what RIF allows, and no more than a step has
    constexpr int U = (CPL >= RIF) ? 1 : (RIF / CPL) * GPW > kMine ? kMine / GPW : RIF / CPL;
    constexpr int C = 64 * KPL;
    const int gl = lane & (G - 1);

    for (;;) {
        int qid = 0;
        if (lane == 0 && part == 0) qid = atomicAdd(a.next_qid, 1);
        if constexpr (WPQ > 1) {
            __syncthreads();  // the query before is done with the workgroup's LDS
            if (threadIdx.x == 0) *s_qid = qid, *s_exact = 0, *s_screened = 0;
            __syncthreads();
            qid = *s_qid;
        }
        qid = __builtin_amdgcn_readfirstlane(qid);
        if (qid >= a.Q) break;

        // a new epoch; the byte wraps after 255 queries of this slot, then the array starts over
        if (!bitmap && ++epoch == 256u) {
            uint4* p = reinterpret_cast<uint4*>(vis);
            for (size_t i = lane; i < b.stride / 16; i += 64) p[i] = make_uint4(0u, 0u, 0u, 0u);
            __threadfence();
            epoch = 1u;
        }
        const uint8_t tag = (uint8_t)epoch;
        for (int i = lane; i < bloom_words; i += 64) bloom[i] = 0u;
        for (int i = lane; i < (tl ? (1 << tl) >> 1 : 0); i += 64) table[i] = 0u;
        for (int i = part * 64 + lane; i < (b.bitmap_words >> 2); i += WPQ * 64) reinterpret_cast<uint4*>(bits)[i] = make_uint4(0u, 0u, 0u, 0u);
        bool any_over = tl == 0;  // has an id of this query gone to the state in HBM?
        uint32_t* visw = reinterpret_cast<uint32_t*>(vis);
        // first visit?  (every lane passes its own id; ids of one call are distinct, or told apart by the caller)
        auto unvisited = [&](uint32_t id) -> bool {
            if (!packed) return __hip_atomic_load(vis + id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != tag;
            const uint32_t w = __hip_atomic_load(visw + id / 24u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return (w >> 24) != epoch || ((w >> (id % 24u)) & 1u) == 0u;
        };
        // Mark a visit.  Packed: bring the word to this epoch (a maximum: words of older epochs lose their flags, a
        // word of this epoch keeps them), then set the flag; both without a return value, and any interleaving of the
        // two operations of several lanes on one word ends with all their flags set.
        auto mark = [&](uint32_t id) {
            if (!packed) {
                __hip_atomic_store(vis + id, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else {
                __hip_atomic_fetch_max(visw + id / 24u, epoch << 24, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_fetch_or(visw + id / 24u, 1u << (id % 24u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        };

        float4 qreg[CPL];
        {
            const float4* q4 = reinterpret_cast<const float4*>(a.queries + (size_t)qid * dim);
#pragma unroll
            for (int t = 0; t < CPL; ++t) {
                const int c = gl + G * t;
                qreg[t] = c < chunks ? q4[c] : make_float4(0, 0, 0, 0);
            }
        }

        // The query in integer codes for the screening on eight-bit rows (search_device.h): bytes in LDS; |q~|^2, the
        // scale and |q - q~| in registers.
        float c_qq = 0.0f, c_sq = 0.0f, c_eq = 0.0f;
        if constexpr (SCREEN == 2) {
            code_query(a.queries + (size_t)qid * dim, dim, lane, qh8, ql8, c_qq, c_sq, c_eq);
            wave_sync();
        }

        uint64_t beam[KPL];
#pragma unroll
        for (int j = 0; j < KPL; ++j) beam[j] = lane * KPL + j < C - L ? kFront : kKeyMax;
        uint64_t live = kKeyMax;  // the worst entry of a full beam
        int nd = 0, ne = 0;
        int n_screened = 0, n_exact = 0, n_vreq = 0;  // rows measured on the smaller copy, fp32 rows, visited-state requests to HBM

        // the lanes with `pass` put their key into the beam
        auto insert_keys = [&](bool pass, uint64_t key) {
            for (uint64_t m = __ballot(pass); m; m &= m - 1) beam_insert<KPL>(beam, readlane_u64(key, __ffsll((long long)m) - 1));
            live = readlane_u64(beam[KPL - 1], 63);
        };
        // The wavefront's share of the list, T of its kMine entries (the others hold some valid id) -> distances -> the
        // beam, or the list of candidates that the wavefronts of a query exchange.
        auto measure_and_merge = [&](int T) {
            const uint32_t* list = todo + part * kMine;
            if constexpr (WPQ > 1) {
                if (lane < kMine) cand[part * kMine + lane] = kKeyMax;
                if (T == 0) return;
                wave_sync();
            }
            // what the screening leaves: lanes with `exact` file their id; entries behind the last hold a valid id
            auto keep = [&](bool exact, int id, int& n2) {
                const uint64_t m = __ballot(exact);
                if (exact) todo2[n2 + prefix_popc(m)] = (uint32_t)id;
                n2 += __popcll(m);
            };
            // Screening (see beam_search.hip): each row is first measured in the half-precision copy of the vectors;
            // a row whose exact distance is certainly beyond the beam's worst entry is dropped without reading its
            // fp32 row -- most of what a search measures once its beam is full.
            if constexpr (SCREEN == 1 && G == 64) {
              if (live != kKeyMax) {
                constexpr int UH = U > kScreenRows ? kScreenRows : U;
                constexpr int RPIH = 2 * UH;
                const int glh = lane & 31, grph = lane >> 5;
                const int chunksH = (dim + 7) >> 3;
                const float s_live = key_s(live);
                // the lane's share of the query: the eight dimensions of each 16-byte chunk of halves it reads
                // (fetched with the rows rather than kept in registers for the whole query)
                float4 qa[CPL][2];
                {
                    const float4* q4 = reinterpret_cast<const float4*>(a.queries + (size_t)qid * dim);
#pragma unroll
                    for (int t = 0; t < CPL; ++t) {
                        const int c = 2 * (glh + 32 * t);
                        qa[t][0] = c < chunks ? q4[c] : make_float4(0, 0, 0, 0);
                        qa[t][1] = c + 1 < chunks ? q4[c + 1] : make_float4(0, 0, 0, 0);
                    }
                }
                int n2 = 0;
                if (lane < kBatch) todo2[lane] = list[0];
                wave_sync();
                for (int base = 0; base < T; base += RPIH) {
                    int vid[UH];
                    const int r0 = base + grph * UH;
#pragma unroll
                    for (int u = 0; u < UH; ++u) vid[u] = r0 + u < T ? (int)list[r0 + u] : -1;
                    uint4 h[UH][CPL];
#pragma unroll
                    for (int u = 0; u < UH; ++u) {
                        const uint4* row = reinterpret_cast<const uint4*>(
                            b.vec16 + (uint64_t)(uint32_t)(vid[u] < 0 ? 0 : vid[u]) * b.stride16);
#pragma unroll
                        for (int t = 0; t < CPL; ++t) {
                            const int c = glh + 32 * t;
                            h[u][t] = (vid[u] >= 0 && c < chunksH) ? row[c] : make_uint4(0u, 0u, 0u, 0u);
                        }
                    }
                    const int mi = r0 + filed_row<32, UH>(lane);
                    const int myid = (glh < UH && mi < T) ? (int)list[mi] : -1;  // the row this lane files
                    const bool valid = myid >= 0;
                    float nx = 0.0f;
                    if (valid)
                        nx = *reinterpret_cast<const float*>(b.vec16 + (uint64_t)(uint32_t)myid * b.stride16 +
                                                             (size_t)chunksH * 16);
                    float acc[UH];
#pragma unroll
                    for (int u = 0; u < UH; ++u) {
                        float sum = 0.0f;
#pragma unroll
                        for (int t = 0; t < CPL; ++t) {
                            const __half2* hp = reinterpret_cast<const __half2*>(&h[u][t]);
                            const float2 x0 = __half22float2(hp[0]), x1 = __half22float2(hp[1]);
                            const float2 x2 = __half22float2(hp[2]), x3 = __half22float2(hp[3]);
                            float d;
                            d = qa[t][0].x - x0.x, sum = __fmaf_rn(d, d, sum);
                            d = qa[t][0].y - x0.y, sum = __fmaf_rn(d, d, sum);
                            d = qa[t][0].z - x1.x, sum = __fmaf_rn(d, d, sum);
                            d = qa[t][0].w - x1.y, sum = __fmaf_rn(d, d, sum);
                            d = qa[t][1].x - x2.x, sum = __fmaf_rn(d, d, sum);
                            d = qa[t][1].y - x2.y, sum = __fmaf_rn(d, d, sum);
                            d = qa[t][1].z - x3.x, sum = __fmaf_rn(d, d, sum);
                            d = qa[t][1].w - x3.y, sum = __fmaf_rn(d, d, sum);
                        }
                        acc[u] = sum;
                    }
                    const float mine = rows_sum<32, UH>(acc);
                    // (2^-11 |x| for components that are normal in half precision, 2^-25 each for smaller ones)
                    const float root = sqrtf(mine), r = 5.0e-4f * nx + 1.0e-6f + 3.0e-8f * sqrtf((float)(chunksH * 8));
                    const float lo_root = fmaxf(root - r, 0.0f);
                    const float lo = lo_root * lo_root * (1.0f - 1.0e-4f);
                    keep(valid && !(lo > s_live), myid, n2);
                }
                wave_sync();
                list = todo2;
                n_screened += T;
                T = n2;
              }
            }
            if constexpr (SCREEN == 2 && G >= 32 && CPL <= 2) {
                if (live != kKeyMax) {
                    // the same on eight-bit codes: sixteen lanes per row, all 32 rows of a step in one round of requests
                    constexpr int CPL8 = CPL;
                    constexpr int U8M = (WGS <= 2 ? 8 : 8 / CPL8) < kMine / 4 ? (WGS <= 2 ? 8 : 8 / CPL8) : kMine / 4;
                    const int gl8 = lane & 15, grp8 = lane >> 4;
                    const int nck = (dim + 15) >> 4;
                    const float s_live = key_s(live);
                    CodedQuery<CPL8> cq;
                    load_coded_query<CPL8>(qh8, ql8, nck, gl8, cq);
                    int n2 = 0;
                    if (lane < kBatch) todo2[lane] = list[0];
                    wave_sync();
                    auto screen_pass = [&](auto rows, int base) {
                        constexpr int U8 = decltype(rows)::value;
                        int vid[U8];
#pragma unroll
                        for (int u = 0; u < U8; ++u) vid[u] = (int)list[base + u * 4 + grp8];
                        const int mi = base + filed_row<16, U8>(lane) * 4 + grp8;
                        const int myid = (gl8 < U8 && mi < T) ? (int)list[mi] : -1;  // the row this lane files
                        float lo, hi;
                        coded_rows_bounds<CPL8, U8>(b.vec8, (uint32_t)b.stride8, nck, gl8, vid, myid, cq, c_qq, c_sq, c_eq, a.metric, lo, hi);
                        keep(myid >= 0 && !(lo > s_live), myid, n2);
                    };
                    for (int base = 0; base < T; base += 4 * U8M) {
                        if (U8M == 8 && T - base <= 16)
                            screen_pass(std::integral_constant<int, (U8M == 8 ? 4 : U8M)>{}, base);
                        else
                            screen_pass(std::integral_constant<int, U8M>{}, base);
                    }
                    wave_sync();
                    list = todo2;
                    n_screened += T;
                    T = n2;
                }
            }
            n_exact += T;
            // As many rows per pass as there are, up to U: no wait of a step is for fewer than it could be.  The last pass reads
            // the first row again in the place of those that are missing; rows of more than 512 floats, of which a pass takes
            // four, take passes of two and of one for that (reading up to three of 4 and 8 KB for nothing in each step cost 2 ..
            // 7 %: 70 000 x 1536, 2000 queries, L = 450: 11.25 -> 10.69 ms).
            constexpr int kQuarterFrom = CPL >= 4 ? 4 : 16, kHalfFrom = CPL >= 4 ? 2 : 8;
            for (int first = 0; first < T; first += U * GPW) {
                const int left = T - first;
                float s;
                int place;
                if (U >= kQuarterFrom && left <= U / 4 * GPW)
                    s = measure_rows<G, CPL, (U >= kQuarterFrom ? U / 4 : U)>(a.vec, list, first, dim, a.metric, qreg, place);
                else if (U >= kHalfFrom && left <= U / 2 * GPW)
                    s = measure_rows<G, CPL, (U >= kHalfFrom ? U / 2 : U)>(a.vec, list, first, dim, a.metric, qreg, place);
                else
                    s = measure_rows<G, CPL, U>(a.vec, list, first, dim, a.metric, qreg, place);
                const bool valid = place < T;
                const uint64_t key = make_key(s, valid ? (int32_t)list[place] : 0, 0u);
                // the queue turns away what is not better than its worst entry once it is full
                // (include/efanna2e/neighbor.h:162-166)
                const bool pass = valid && s < 3.402823466e+38f && key < live;
                if constexpr (WPQ > 1) {
                    if (pass) cand[part * kMine + place] = key;
                } else {
                    insert_keys(pass, key);
                }
            }
        };

        // ---- the seeds, up to 32 at a time: every start id is visited and measured (src/search_in_cpu.cpp:74-79); then
        // one expansion per step.  (One loop for both, so that the code of a step is there once.)
        bool marked = false;  // marks of this wavefront in HBM that later loads must see
        int seeds_left = M, turn = 0;
        if constexpr (WPQ > 1) __syncthreads();  // the bitmap is clear
        for (;;) {
            int v = -1;
            const bool seeding = seeds_left > 0;
            if (seeding) {
                if (part == 0 && lane < min(seeds_left, kBatch)) v = a.start_ids[M - seeds_left + lane];
                seeds_left -= kBatch;
            } else {
                // the closest entry not yet expanded: the first lane that holds one, the first of its keys
                uint32_t flags = (uint32_t)beam[0];
#pragma unroll
                for (int j = 1; j < KPL; ++j) flags &= (uint32_t)beam[j];
                const uint64_t open = __ballot((flags & 1u) == 0u);
                if (open == 0ull) break;
                const int owner = __ffsll((long long)open) - 1;
                int jj = KPL - 1;
                uint32_t elo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)beam[KPL - 1], owner);
#pragma unroll
                for (int j = KPL - 2; j >= 0; --j) {
                    const uint32_t x = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)beam[j], owner);
                    if ((x & 1u) == 0u) elo = x, jj = j;
                }
                const uint32_t eid = elo >> 1;
                if (lane < R && part == 0) v = a.nbrs[(size_t)eid * R + lane];
                const uint64_t flag = lane == owner ? 1ull : 0ull;
#pragma unroll
                for (int j = 0; j < KPL; ++j) beam[j] |= jj == j ? flag : 0ull;
                ++ne;
            }

            // The tags written in the step before are read by this step through other lanes.  Tag loads and stores are
            // agent-scope atomics, so both go to L2 past the CU's cache; the fence makes the wavefront wait for its
            // stores to be acknowledged (beside the graph row, which it waits for anyway) before it issues the loads
            // below.  (A fence of agent scope would also write the whole L2 back each step, which no other wavefront
            // needs: slots are private.)
            if (marked) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            bool isnew = false, over = false, tested = false;
            if (bitmap) {
                // one atomic per id settles the test, repeated ids of a row included
                if (v >= 0) isnew = ((atomicOr(&bits[(uint32_t)v >> 5], 1u << (v & 31)) >> (v & 31)) & 1u) == 0u;
            } else {
                if (!b.rows_unique) {
                    // an id listed twice in the row counts once (the first listing)
                    const int v0 = v;
                    for (int k = 0; k < R; ++k) {
                        const int vk = __builtin_amdgcn_readlane(v0, k);
                        if (k < lane && vk == v0) v = -1;
                    }
                }
                // the table first; what it has no room for is settled against the state in HBM, which holds nothing
                // before the first id went there, and whose filter knows every id that did
                if (v >= 0) {
                    if (tl) {
                        const int r = table_test_and_set((uint32_t)v);
                        isnew = r == 1, over = r == 2;
                    } else {
                        over = true;
                    }
                    if (over) {
                        const bool settled = seeding || !any_over || (bl && !bloom_may_hold((uint32_t)v));
                        isnew = settled || unvisited((uint32_t)v);
                        tested = !settled;
                    }
                }
                if (isnew && over) {
                    mark((uint32_t)v);
                    if (bl) bloom_add((uint32_t)v);
                }
                const uint64_t mo = __ballot(isnew && over);
                n_vreq += __popcll(__ballot(tested)) + __popcll(mo) * (packed ? 2 : 1);
                marked = mo != 0ull;
                any_over = any_over || marked;
            }
            const uint64_t m = __ballot(isnew);
            int T = __popcll(m);
            if (T != 0) {
                // entries behind the last new id repeat the first: a pass of rows needs no bounds
                const int pad = __builtin_amdgcn_readlane(v, __ffsll((long long)m) - 1);
                if (lane < kBatch) todo[lane] = (uint32_t)pad;
                wave_sync();
                const int rank = prefix_popc(m);
                if (isnew) todo[rank % WPQ * kMine + rank / WPQ] = (uint32_t)v;
                wave_sync();
            }
            if constexpr (WPQ > 1) {
                // (two counts in turn: the first wavefront may be a barrier ahead, and no more, of one that reads)
                if (threadIdx.x == 0) s_new[turn] = T;
                __syncthreads();
                T = __builtin_amdgcn_readfirstlane(s_new[turn]);
                turn ^= 1;
            }
            nd += T;
            if (T == 0) continue;
            measure_and_merge((T - part + WPQ - 1) / WPQ);
            if constexpr (WPQ > 1) {
                __syncthreads();
                // (the next step's candidates are written behind the barrier above, which the next step passes first)
                const uint64_t key = lane < kBatch ? cand[lane] : kKeyMax;
                insert_keys(key < live, key);
            }
            wave_sync();
        }

        // ---- output: the k closest live entries, closest first
        if constexpr (WPQ > 1) {
            if (lane == 0) atomicAdd(s_exact, n_exact), atomicAdd(s_screened, n_screened);
            __syncthreads();
            if (part != 0) continue;
            n_exact = *s_exact, n_screened = *s_screened;
        }
        {
            int32_t* ids_out = a.ids_out + (size_t)qid * a.k;
            float* dists_out = a.dists_out ? a.dists_out + (size_t)qid * a.k : nullptr;
            uint32_t livee = 0;  // bit j: key j of this lane is an entry that is not deleted
#pragma unroll
            for (int j = 0; j < KPL; ++j) {
                if (beam[j] == kFront || beam[j] == kKeyMax) continue;
                bool keep = true;
                if (a.deleted) {
                    const int32_t id = key_id(beam[j]);
                    keep = ((a.deleted[id >> 5] >> (id & 31)) & 1u) == 0;
                }
                livee |= keep ? 1u << j : 0u;
            }
            const int mine = __popc(livee), upto = wave_inclusive_sum(mine);
            const int outpos = __builtin_amdgcn_readlane(upto, 63);
            int pos = upto - mine;
#pragma unroll
            for (int j = 0; j < KPL; ++j) {
                if (((livee >> j) & 1u) == 0u) continue;
                if (pos < a.k) {
                    ids_out[pos] = key_id(beam[j]);
                    if (dists_out) {
                        const float s = key_s(beam[j]);
                        dists_out[pos] = a.metric == 0 ? s : 0.0f - s;
                    }
                }
                ++pos;
            }
            for (int i = outpos + lane; i < a.k; i += 64) {
                ids_out[i] = -1;
                if (dists_out) {
                    const float far = __int_as_float(0x7f800000);  // src/search_in_cpu.cpp:33-35
                    dists_out[i] = a.metric == 0 ? far : -far;
                }
            }
            if (lane == 0) {
                int32_t* c = a.counters + (size_t)qid * 4;
                c[0] = M + ne, c[1] = ne, c[2] = nd, c[3] = ne;
                {
                    int32_t* rc = a.counters + ((size_t)a.Q + qid) * 4;
                    rc[0] = n_screened, rc[1] = n_exact, rc[2] = 0, rc[3] = n_vreq;
                }
            }
        }
        if (marked) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        wave_sync();
    }
    if (!bitmap && lane == 0) b.epochs[slot] = epoch;
}

}  // namespace
}  // namespace coral
