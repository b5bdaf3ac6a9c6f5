// best_first_shared.hip -- the best-first kernel (best_first_device.h) with four wavefronts per query, which share the
// rows of a step: for a few queries on wide rows.
#include "best_first_device.h"

namespace coral {

namespace {

using bf_kernel_fn = void (*)(const SearchArgs, const BestFirstArgs);

template <int KPL, int SCREEN>
bf_kernel_fn pick_shared_width(int chunks) {
    if (chunks <= 64) return best_first_wave_kernel<64, 1, 8, KPL, SCREEN, 2, 4>;
    if (chunks <= 128) return best_first_wave_kernel<64, 2, 16, KPL, SCREEN, 2, 4>;
    if constexpr (SCREEN == 0) {  // (rows of more than 512 floats have no copy in eight-bit codes)
        if (chunks <= 256) return best_first_wave_kernel<64, 4, 32, KPL, SCREEN, 2, 4>;
        if (chunks <= 512) return best_first_wave_kernel<64, 8, 32, KPL, SCREEN, 2, 4>;
    }
    return nullptr;
}

template <int SCREEN>
bf_kernel_fn pick_shared(int dim, int L) {
    if (L <= 128) return pick_shared_width<2, SCREEN>(dim / 4);
    if (L <= 256) return pick_shared_width<4, SCREEN>(dim / 4);
    if (L <= 512) return pick_shared_width<8, SCREEN>(dim / 4);
    if (L <= 1024) return pick_shared_width<16, SCREEN>(dim / 4);
    if (L <= 1280) return pick_shared_width<20, SCREEN>(dim / 4);
    return nullptr;
}

}  // namespace

size_t best_first_shared_lds_bytes(int coded_bytes, int bitmap_words) {
    return kSharedStepBytes + best_first_wave_lds_bytes(0, 0, coded_bytes, bitmap_words);
}

hipError_t best_first_shared_prepare(int dim, int L, int screen, size_t lds, int* max_wg_per_cu) {
    if (screen == 1 || (screen == 2 && dim > kMaxByteRowDim)) return hipErrorInvalidValue;
    bf_kernel_fn fn = screen == 2 ? pick_shared<2>(dim, L) : pick_shared<0>(dim, L);
    if (!fn) return hipErrorInvalidValue;
    hipError_t e = raise_lds_limit(reinterpret_cast<const void*>(fn), lds);
    if (e != hipSuccess) return e;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(max_wg_per_cu, reinterpret_cast<const void*>(fn), kWavesPerWg * 64, lds);
}

hipError_t launch_best_first_shared(const SearchArgs& a, const BestFirstArgs& b, hipStream_t stream) {
    const int screen = b.vec8 != nullptr ? 2 : 0;
    if (screen == 2 && (a.dim > kMaxByteRowDim || b.coded_bytes != coded_query_bytes(a.dim))) return hipErrorInvalidValue;
    if (a.R > kBatch || a.M <= 0 || b.slots <= 0 || b.table_log2 != 0 || b.bloom_log2 != 0 || b.vec16 != nullptr) return hipErrorInvalidValue;
    if ((b.bitmap_words & 3) != 0 || (int64_t)b.bitmap_words * 32 < a.n) return hipErrorInvalidValue;
    bf_kernel_fn fn = screen == 2 ? pick_shared<2>(a.dim, a.L) : pick_shared<0>(a.dim, a.L);
    if (!fn) return hipErrorInvalidValue;
    hipLaunchKernelGGL(fn, dim3(b.slots), dim3(kWavesPerWg * 64), best_first_shared_lds_bytes(b.coded_bytes, b.bitmap_words), stream, a, b);
    return hipGetLastError();
}

}  // namespace coral
