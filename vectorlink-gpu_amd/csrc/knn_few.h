// Exact kNN of a few queries (knn_few.hip), as knn.hip uses it.
#pragma once
#include "vl_common.h"

// Whether a batch goes to the kernel of knn_few.hip.  Its time grows with every 32 queries and with the table; the filter
// of knn_filter.hip takes the larger batches, at some 70 us and more for its launches (us, this kernel / the filter, k = 4):
// 32,768 x 64: 128 queries 41 / 73; 32,768 x 768: 64: 83 / 137, 128: 147 / 137; 200,000 x 128: 64: 104 / 133, 128: 177 / 133;
// 500,000 x 768: 32: 527 / 835, 33: 1,168 / 835.  (The float32 tiles, which take calls that are too short for the
// filter, cost the same for 1 query as for 128: 234 at 32,768 x 768.)
inline bool vl_knn_is_few(int64_t n_queries, int64_t n_vectors, int64_t dim) {
    const int64_t most = n_vectors * dim <= (8ll << 20) ? 128 : (n_vectors * dim <= (32ll << 20) ? 64 : 32);
    return n_queries <= most;
}

// Lists of list_len keys that the kernel keeps per query for a table of this size.
int64_t vl_knn_few_lists(int64_t n_vectors);
int vl_knn_few(const float *queries, int64_t n_queries, const float *vectors, int64_t n_vectors, int64_t dim, int64_t k,
               int list_len, bool l2, const float *q_norm, const float *v_norm, uint64_t *cand, int32_t *ids_out,
               float *dists_out, hipStream_t st);
