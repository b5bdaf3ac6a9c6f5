// bruteforce.h -- host-side launchers of the exact kNN kernels (bruteforce.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace coral {
hipError_t launch_distance_tile(const float* queries, const float* base, int nq, int64_t nb, int dim,
                                int metric, const uint32_t* deleted, int64_t base_id0, float* D,
                                int64_t ldD, hipStream_t stream);
// tau: only the value of the k-th smallest of every row (+inf if there are fewer); out is not written then
// redo: int[nq] scratch for the rows the fast path hands over (null: radix path for every row)
hipError_t launch_row_select(const float* D, int64_t ldD, int nq, int64_t n, int k, int64_t id0,
                             unsigned long long* out, int64_t out_stride, int* redo, hipStream_t stream,
                             float* tau = nullptr);
hipError_t launch_merge_segments(const unsigned long long* part, int nq, int nseg, int k, int metric,
                                 int32_t* ids, float* dists, hipStream_t stream);
// --- the screening pass on the matrix cores (bruteforce_mfma.hip) ---
// out[r] (optional) = |x_r|^2; *max_bits (optional, zero before) = bit pattern of the largest of them; *res_max (optional):
// the same for a bound on |x_r - hi(x_r)|, what one half per component leaves out
hipError_t launch_row_norms(const float* x, int64_t n, int dim, float* out, uint32_t* max_bits, uint32_t* res_max,
                            hipStream_t stream);
// the queries in the form the two launches below take them (split into halves, tile by tile) into out (that many bytes),
// qn[q] = |q|^2, and, where given, res[q] = that bound, cnt[q * kCntStride] = 0, zero[0] = zero[1] = 0.
// products: 3 (hi.hi + hi.lo + lo.hi, about fp32 accuracy) or 1 (hi.hi alone), the same in all launches of a call
size_t split_queries_bytes(int nq, int dim, int products);
size_t split_queries_offset(int64_t row, int dim, int products);  // of a row that is a multiple of kQueryTile
constexpr int kQueryTile = 256;
// ints of an index's pinned memory for what a call reads back: the flags of 1024 queries and one more (4 KB over the bus)
constexpr int kKnnFlags = 1025;
hipError_t launch_prepare_queries(const float* queries, int nq, int dim, int products, float* qn, float* res, void* out,
                                  unsigned int* cnt, int* zero, hipStream_t stream);
// as launch_distance_tile, with D[q][b] = |q|^2 + |b|^2 - 2 q.b (L2) or -q.b (IP) from inner products on the matrix
// cores; queries: what launch_prepare_queries wrote.
// sample_tiles > 0: only that many tiles of 128 base points, every tile_stride-th of the base, side by side in D
hipError_t launch_approx_tile(const void* queries, const float* base, int nq, int64_t nb, int dim, int metric, int products,
                              const float* qn, const float* bn, const uint32_t* deleted, int64_t base_id0, float* D,
                              int64_t ldD, hipStream_t stream, int64_t sample_tiles = 0, int tile_stride = 1);
// the same distances, no matrix: every entry <= tau[q] is appended to lists[q * cap ...] as ord(value) << 32 | id
// (cnt[q * kCntStride] counts them, also those beyond cap that were dropped).  tile_step > 0: tiles 0, tile_step,
// 2 tile_step ... of 128 base points; tile_step < 0: the tiles between those
constexpr int kCntStride = 16;  // a 64-byte line per counter: workgroups append to many queries at a time
hipError_t launch_approx_filter(const void* queries, const float* base, int nq, int64_t nb, int dim, int metric, int products,
                                const float* qn, const float* bn, const uint32_t* deleted, const float* tau,
                                unsigned long long* lists, int64_t cap, unsigned int* cnt, int tile_step,
                                hipStream_t stream);
// the k (<= 1024) smallest keys of every list, sorted, as ids [nq][k] (-1: none) and values; *overflow (zero before)
// counts the lists that could not be done; their ids are -1
hipError_t launch_list_select(unsigned long long* lists, int64_t cap, unsigned int* cnt, int nq, int k, int32_t* ids,
                              float* dists, int* overflow, hipStream_t stream);
// the same selection in place, between two launches that append: the list shrinks to its k smallest keys, tau[q]
// becomes the value of the k-th (and stays what it was if there are fewer)
hipError_t launch_list_shrink(unsigned long long* lists, int64_t cap, unsigned int* cnt, int nq, int k, float* tau,
                              int* overflow, hipStream_t stream);
// cand_ids / cand_d [nq][kc] (ascending approximate signed distance, -1 = none) -> the exact k best per query in the
// reference's summation order; redo[q] = 1 where the candidates cannot vouch for the result,
// redo[nq] = *lost (null: 0)
hipError_t launch_rerank(const float* queries, const float* base, int nq, int dim, int metric, const int32_t* cand_ids,
                         const float* cand_d, int kc, int k, const float* qn, const uint32_t* bn_max_bits, const float* qres,
                         const uint32_t* bres_max_bits, int32_t* ids, float* dists, int* redo, const int* lost, hipStream_t stream);
// (qres, *bres_max_bits: what launch_prepare_queries and launch_row_norms gave, for candidates chosen on one product; else null)
// *extra += the entries of D's rows, beyond kc, that one product cannot tell from those up to tau
hipError_t launch_count_close(const float* D, int64_t ldD, int nq, int64_t n, int kc, int metric, const float* qn,
                              const uint32_t* bn_max_bits, const float* qres, const uint32_t* bres_max_bits, const float* tau,
                              int* extra, hipStream_t stream);
// --- levels: four bits per (query, base point) that bound the distance from below and above (bruteforce_mfma.hip) ---
// Level l in 0 .. 14 of an entry means: its exact signed distance lies in [origin + l step - E, origin + (l + 1) step + E],
// the lower end void for l = 0 and the upper one for l = 0 and l = 14; ranges[q] = origin, 1 / step, step, E (1 / step = 0: all
// levels are 0).  Point i of query q: bits 4 (i & 1) of byte levels[q * level_pitch(n) + i / 2].
size_t level_pitch(int64_t n);
// D: [nq][n] approximate distances to a sample of the base, made on one product; unfit: null, or a word that grows by the
// queries whose levels would settle little
hipError_t launch_level_ranges(const float* D, int64_t ldD, int nq, int n, int dim, int metric, const float* qn,
                               const uint32_t* bn_max_bits, const float* qres, const uint32_t* bres_max_bits, float4* ranges,
                               int* unfit, hipStream_t stream);
// queries: split for one product
hipError_t launch_levels(const void* queries, const float* base, int nq, int64_t nb, int dim, int metric, const float* qn,
                         const float* bn, const float4* ranges, unsigned char* levels, hipStream_t stream);
hipError_t launch_scatter_results(const int32_t* rows, int count, int k, const int32_t* src_ids, const float* src_d,
                                  int32_t* dst_ids, float* dst_d, hipStream_t stream);
}  // namespace coral
