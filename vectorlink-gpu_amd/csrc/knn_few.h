// Exact kNN of a few queries (knn_few.hip), as knn.hip uses it.
#pragma once
#include "vl_common.h"

// Most queries that go to the kernel of knn_few.hip.  Its time grows with every 32 of them, a tile of knn.hip costs the
// same for 1 as for 128 (us, this kernel / tiles; k = 4): 32,768 x 768: 1 query 43 / 234, 64: 83 / 250, 128: 147 / 255,
// 256: 278 / 255; 500,000 x 768: 1: 463 / 3,094, 128: 2,162 / 3,149, 256: 4,204 / 3,160.
constexpr int64_t kFewQueries = 128;

// Lists of list_len keys that the kernel keeps per query for a table of this size.
int64_t vl_knn_few_lists(int64_t n_vectors);
int vl_knn_few(const float *queries, int64_t n_queries, const float *vectors, int64_t n_vectors, int64_t dim, int64_t k,
               int list_len, bool l2, const float *q_norm, const float *v_norm, uint64_t *cand, int32_t *ids_out,
               float *dists_out, hipStream_t st);
