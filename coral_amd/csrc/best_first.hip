// best_first.hip -- the best-first traversal (the reference's CPU search, src/search_in_cpu.cpp:63-108) with one
// WAVEFRONT per in-flight query.
//
// Best-first expands one beam entry at a time: read its graph row, test its neighbours against the visited set,
// measure the new ones, insert them, pick the closest entry not yet expanded.  Every step is a chain of dependent
// waits and of instructions that a lone wavefront issues one after the other; what makes it fast on this GPU is how
// short that chain is and how many such chains run side by side.
//
// The sorted beam lives in the wavefront's registers, KPL consecutive keys per lane (L = 512: 16 registers): a key is
// inserted by one exchange with the lane below and five instructions per place, and the next entry to expand is found
// by a ballot.  The beam in LDS, as it was, cost ranks, binary searches, byte counters and shifted copies: of the 10 000
// cycles of a step on 96-float rows (L = 100, a wavefront per SIMD) 2800, now 1200; 97 queries on 50 001 x 96: 610 ->
// 350 us.  LDS holds the visited set instead.
//
// The visited set.  Where the wavefronts that a batch gives a CU find LDS for it, a bitmap of all ids: one atomic per
// id.  Else it has two levels.  In global memory, the form the CPU path itself uses (src/search_in_cpu.cpp:44-48,
// 68-71): one byte per node and query slot holding the epoch of the query that last visited the node, so nothing
// is cleared between queries (every 255th query of a slot wipes its array).  With 288 GB of HBM four thousand such
// arrays are cheap (4 GB at a million nodes); each test costs a 128-byte line of HBM traffic and each mark a
// 32-byte write.  For indexes too large for a byte per node and slot the same state is packed into 32-bit words of
// 8 epoch bits over 24 node flags.  A Bloom filter over the query's visited ids in LDS (8 KB at L = 512) answers most
// tests without that line: an id it does not know is new for certain.
// Those single-line requests cost the memory system more than their bytes say, so where the beam is short enough --
// 8192 cells hold a query's visits up to L = 409 -- the first level is an exact table of 16-bit cells in LDS, in buckets
// of four with two candidate buckets per id: a test is two 8-byte LDS reads whatever the load, and only ids that find
// both buckets full go to the state in HBM.
//
// Rows of more than 128 floats are screened on their eight-bit codes.  4999 queries on 250 000 x 200 at L = 512 (a full
// chip and a second pass): 6.2 -> 4.9 ms.  Over 252 launches (six graphs, L = 32 .. 1000, 1 .. 5000 queries) the time is 0.58 of
// what it was with the beam in LDS, geometric mean.
//
// The arithmetic is that of beam_search.hip (same lane-strided accumulation, same butterfly, same 64-bit keys), so
// results and counters are identical bit for bit; a wavefront needs no workgroup barrier anywhere.
#include "best_first_device.h"

namespace coral {

namespace {

// one thread per graph row: does it list an id twice?
__global__ __launch_bounds__(256) void find_repeated_ids_kernel(const int32_t* __restrict__ nbrs, int64_t n, int R,
                                                                uint32_t* flag) {
    const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= n) return;
    const int32_t* r = nbrs + row * R;
    bool rep = false;
    for (int i = 1; i < R; ++i) {
        const int32_t v = r[i];
        if (v < 0) break;  // rows end at their first -1
        for (int j = 0; j < i; ++j) rep |= r[j] == v;
    }
    if (rep) atomicOr(flag, 1u);
}

using bf_kernel_fn = void (*)(const SearchArgs, const BestFirstArgs);

// The form for a row width: G lanes per row, CPL chunks per lane.  Rows of more than 512 floats have no copy in
// eight-bit codes, rows of up to 128 no other, rows of up to 64 none: what no launch asks for is not built.
template <int RIF, int KPL, int SCREEN, int WGS>
bf_kernel_fn pick_bf_width(int chunks) {
    // (what fits the registers beside the beam without spilling two dozen of them)
    constexpr int RIF4 = WGS > 2 && KPL >= 8 ? 8 : RIF, RIF8 = WGS > 2 ? 8 : RIF;
    if constexpr (SCREEN == 0) {
        if (chunks <= 16) return best_first_wave_kernel<16, 1, (RIF > 16 ? 16 : RIF), KPL, 0, WGS, 1>;
    }
    if constexpr (SCREEN != 1) {
        if (chunks <= 32) return chunks > 16 ? best_first_wave_kernel<32, 1, (RIF > 16 ? 16 : RIF), KPL, SCREEN, WGS, 1> : nullptr;
    }
    if (chunks <= 32) return nullptr;
    if (chunks <= 64) return best_first_wave_kernel<64, 1, RIF, KPL, SCREEN, WGS, 1>;
    if (chunks <= 128) return best_first_wave_kernel<64, 2, RIF, KPL, SCREEN, WGS, 1>;
    if constexpr (SCREEN != 2) {
        if (chunks <= 256) return best_first_wave_kernel<64, 4, RIF4, KPL, SCREEN, WGS, 1>;
        if (chunks <= 512) return best_first_wave_kernel<64, 8, RIF8, KPL, SCREEN, WGS, 1>;
    }
    return nullptr;
}

// rif: 32 for launches that hold eight wavefronts per CU or fewer (256 registers per lane); 16, and with a screening,
// which leaves few rows of a step to read in fp32, 8 otherwise.  The registers of a lane must hold its share of the
// beam beside the rows: sixteen wavefronts per CU up to L = 512, twelve up to 1280, eight beyond.
template <int SCREEN>
bf_kernel_fn pick_bf_length(int dim, int rif, int L) {
    const int chunks = dim / 4;
    if constexpr (SCREEN == 0) {
        if (rif >= 32) {
            if (L <= 128) return pick_bf_width<32, 2, 0, 2>(chunks);
            if (L <= 256) return pick_bf_width<32, 4, 0, 2>(chunks);
            if (L <= 512) return pick_bf_width<32, 8, 0, 2>(chunks);
            if (L <= 1024) return pick_bf_width<32, 16, 0, 2>(chunks);
        }
        if (L <= 128) return pick_bf_width<16, 2, 0, 4>(chunks);
        if (L <= 256) return pick_bf_width<16, 4, 0, 4>(chunks);
        if (L <= 512) return pick_bf_width<16, 8, 0, 4>(chunks);
        if (L <= 1024) return pick_bf_width<16, 16, 0, 3>(chunks);
        if (L <= 1280) return pick_bf_width<16, 20, 0, 3>(chunks);
        if (L <= kMaxWaveBeam) return pick_bf_width<16, 32, 0, 2>(chunks);
    } else {
        if constexpr (SCREEN == 2) {
            if (rif >= 32) {
                if (L <= 128) return pick_bf_width<32, 2, SCREEN, 2>(chunks);
                if (L <= 256) return pick_bf_width<32, 4, SCREEN, 2>(chunks);
                if (L <= 512) return pick_bf_width<32, 8, SCREEN, 2>(chunks);
                if (L <= 1024) return pick_bf_width<32, 16, SCREEN, 2>(chunks);
            }
            if (L <= 128) return pick_bf_width<8, 2, SCREEN, 4>(chunks);
            if (L <= 256) return pick_bf_width<8, 4, SCREEN, 4>(chunks);
        }
        if (L <= 512) return pick_bf_width<8, 8, SCREEN, 4>(chunks);
        if (L <= 1024) return pick_bf_width<8, 16, SCREEN, 3>(chunks);
        if (L <= 1280) return pick_bf_width<8, 20, SCREEN, 3>(chunks);
        if (L <= kMaxWaveBeam) return pick_bf_width<8, 32, SCREEN, 2>(chunks);
    }
    return nullptr;
}

bf_kernel_fn pick_bf_kernel(int dim, int rif, int screen, int L) {
    return screen == 2   ? pick_bf_length<2>(dim, rif, L)
           : screen == 1 ? pick_bf_length<1>(dim, rif, L)
                         : pick_bf_length<0>(dim, rif, L);
}

}  // namespace

hipError_t best_first_prepare(int dim, int L, int rows_in_flight, int screen, size_t wave_lds, int* max_wg_per_cu) {
    if (screen == 2 && dim > kMaxByteRowDim) return hipErrorInvalidValue;
    const size_t lds = wave_lds * kWavesPerWg;
    bf_kernel_fn fn = pick_bf_kernel(dim, rows_in_flight, screen, L);
    if (!fn) return hipErrorInvalidValue;
    hipError_t e = raise_lds_limit(reinterpret_cast<const void*>(fn), lds);
    if (e != hipSuccess) return e;
    int nb = 0;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, reinterpret_cast<const void*>(fn), kWavesPerWg * 64, lds);
    if (e != hipSuccess) return e;
    *max_wg_per_cu = nb;
    return hipSuccess;
}

hipError_t launch_best_first(const SearchArgs& a, const BestFirstArgs& b, hipStream_t stream) {
    const int screen = b.vec8 != nullptr ? 2 : b.vec16 != nullptr ? 1 : 0;
    if (screen == 2 && (a.dim > kMaxByteRowDim || b.coded_bytes != coded_query_bytes(a.dim))) return hipErrorInvalidValue;
    if (a.R > kBatch || a.M <= 0 || b.waves_per_wg < 1 || b.waves_per_wg > kWavesPerWg) return hipErrorInvalidValue;
    if (b.bitmap_words != 0 && ((b.bitmap_words & 3) != 0 || (int64_t)b.bitmap_words * 32 < a.n)) return hipErrorInvalidValue;
    const size_t lds = best_first_wave_lds_bytes(b.bloom_log2, b.table_log2, b.coded_bytes, b.bitmap_words) * b.waves_per_wg;
    bf_kernel_fn fn = pick_bf_kernel(a.dim, b.rows_in_flight, screen, a.L);
    if (!fn) return hipErrorInvalidValue;
    const int wgs = (b.slots + b.waves_per_wg - 1) / b.waves_per_wg;
    hipLaunchKernelGGL(fn, dim3(wgs), dim3(b.waves_per_wg * 64), lds, stream, a, b);
    return hipGetLastError();
}

hipError_t launch_find_repeated_ids(const int32_t* nbrs, int64_t n, int R, uint32_t* flag, hipStream_t stream) {
    const int64_t blocks = (n + 255) / 256;
    if (blocks <= 0 || blocks > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL(find_repeated_ids_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, nbrs, n, R, flag);
    return hipGetLastError();
}

}  // namespace coral
