// Dot products of all queries and vectors of a call in bfloat16, kept in 16 bits, and the bounds of a distance that one of them
// gives.  A batch of a first optimisation loop on a table that is too large for all its distances in float32 (beam_table.hip)
// looks its candidates up here instead of fetching their 8-bit sketch: 2 bytes, mostly on a cache line with other
// candidates (PairColumns), instead of a row of dim bytes.  As with the sketch (sketch_device.h), nothing that is returned is
// computed from these values: they tell which candidates cannot enter a queue, and the others are evaluated in float32.
//
// With q^, v^ the rows rounded to bfloat16, | <q, v> - <q^, v^> | <= ||q - q^|| ||v|| + ||q^|| ||v - v^|| (Cauchy-Schwarz), and the
// float32 sums on either side are off by dim 2^-23 of the product of the norms at most; a value is rounded once more, to half.
#pragma once
#include "pair_table.h"
#include "sketch_device.h"

struct NearQuery {
    float per_resid, per_norm;  // the bound's parts for each unit of a vector's residual and norm
};

struct NearPlan {
    int64_t kp, columns;  // columns of a bfloat16 row and of the table: vectors in the order of PairColumns, whole tiles of 256
    int64_t off_queries, off_columns, off_q16, off_v16, off_values, bytes;
};
NearPlan vl_near_plan(int64_t n_queries, int64_t n_vectors, int64_t dim);
// ws: plan.bytes bytes, 256-byte aligned.  Rows are 16-byte aligned, dim a multiple of 4.  Nothing is allocated or waited for.
int vl_launch_near_products(const NearPlan &plan, const float *queries, int64_t n_queries, const float *vectors, int64_t n_vectors,
                            int64_t dim, uint8_t *ws, hipStream_t st);

// lo <= d <= hi for the float32 distance d (dist_device.h).  column: half resid >= ||v - v^||, half norm >= ||v||.
__device__ __forceinline__ void near_bounds(uint32_t value, uint32_t column, const NearQuery &q, float *lo, float *hi) {
    const float s = half_bits_as_float(value);
    const float resid = half_bits_as_float(column & 0xffffu), norm = half_bits_as_float(column >> 16);
    // 5e-4: half of a half's last place, relative; 1e-6: its smallest numbers, and the float operations here and in the map to d
    const float eps = (q.per_resid * resid + q.per_norm * norm + 5e-4f * fabsf(s)) * 1.0001f + 1e-6f;
    const bool known = eps == eps && fabsf(s) < 60000.0f;  // (beyond: an infinity of a half, or no number)
    *lo = known ? clamp_distance(s + eps) : 0.0f;
    *hi = known ? clamp_distance(s - eps) : 1.0f;
}
