// Exact kNN through a bfloat16 filter (knn_filter.hip), as knn.hip uses it.
#pragma once
#include "vl_common.h"

struct KnnFilterPlan {
    int64_t kp;             // columns of a bfloat16 row: dim (and three more for L2) padded to a multiple of 64
    int64_t sample_rows;    // rows of the sample that bounds are taken from (whole tiles)
    int64_t sample_stride;  // between the places of two rows of the sample that follow each other in the table
    int sample_strips;
    int groups;             // maxima per query that the sample pass leaves
    int most;               // candidates of a query that cost what the tiles do for it
    int64_t slab_rows;      // rows of the table converted at a time
    int64_t off_q16, off_v16, off_qstat, off_gmax, off_bound, off_count, off_found, off_vmax, bytes;
};

// Whether a call is taken by the filter, and its plan, which also serves a call of fewer queries.
bool vl_knn_filter_plan(int64_t n_queries, int64_t n_vectors, int64_t dim, int64_t k, bool l2, KnnFilterPlan *p);

// Writes the answers of every query whose candidates are few enough; appends the others to left: left[0] is how many there
// are, their numbers (q_first + place in this call) follow in order.  tile_bound[i] is set for the i-th of them.  A call
// with q_first == 0 starts the list.  ws: p.bytes bytes, 256-byte aligned.  q_norm / v_norm: squared lengths (written here
// when l2, else not used).
int vl_knn_filter(const KnnFilterPlan &p, const float *queries, int64_t n_queries, const float *vectors, int64_t n_vectors,
                  int64_t dim, int64_t k, bool l2, float *q_norm, float *v_norm, int64_t q_first, int32_t *left,
                  uint32_t *tile_bound, char *ws, int32_t *ids_out, float *dists_out, hipStream_t st);
