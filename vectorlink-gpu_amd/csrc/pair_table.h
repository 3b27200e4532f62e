// Distances of all pairs of a batch of queries and a table of vectors, with the bits of dist_device.h (pair_table.hip).
#pragma once
#include "vl_common.h"

// Operands are multiplied from copies in the order in which the sums take them up: 32 vectors make a strip, a strip is a
// row of units of 1 KiB.  A unit belongs to a pair of partial sums (c, c + sums / 2), which the first fold adds; the j-th unit
// of a pair holds chunk c + sums j of the strip's vectors and chunk c + sums / 2 + sums j (zeros past a row's end): lanes
// 0 .. 31 have elements 0 and 2 of both, lanes 32 .. 63 elements 1 and 3.  Pairs come in the order in which the further
// folds can be done as soon as both of their sides are there: the bits of the pair's number reversed.
// sums: 64 partial sums, or as many (a power of two from 16) as rows of few chunks have.
struct PairUnits {
    int sums, nchunks, count;  // count: units of a strip
    int pitch;                 // units from one strip to the next: whole stages (what lies between is read and not used)
};
constexpr int kPairStage = 4;
// units of pair c
__host__ __device__ inline int pair_units_of(int nchunks, int sums, int c) { return c < nchunks ? (nchunks - c + sums - 1) / sums : 0; }
__host__ __device__ inline PairUnits pair_units(int64_t dim) {
    PairUnits u;
    u.nchunks = (int)((dim + 3) / 4);
    u.sums = u.nchunks <= 16 ? 16 : u.nchunks <= 32 ? 32 : 64;
    const int whole = u.nchunks / u.sums, rest = u.nchunks % u.sums;
    u.count = whole * (u.sums / 2) + (rest < u.sums / 2 ? rest : u.sums / 2);
    u.pitch = (u.count + kPairStage - 1) / kPairStage * kPairStage;
    return u;
}

constexpr int kPairTile = 64;    // queries and vectors of a workgroup's tile
constexpr int kPairStrip = 32;   // vectors of a strip
constexpr int64_t kPairUnit = 1024;

// Columns of the table: vectors whose ids are the same modulo 6 stand together.  The neighbours of a node of the circulant
// graph are its id plus primes, which are 1 or 5 modulo 6, so the 128 that it has within 2,000 ids lie on 22 cache lines
// instead of 56 (mean over the nodes of 20,011).
constexpr int kPairClasses = 6;
struct PairColumns {
    uint32_t per_class;
    __host__ __device__ explicit PairColumns(int64_t n_vectors) : per_class((uint32_t)((n_vectors + kPairClasses - 1) / kPairClasses)) {}
    __host__ __device__ uint32_t of(uint32_t id) const { return id % kPairClasses * per_class + id / kPairClasses; }
    __host__ __device__ int64_t vector_at(int64_t column) const {  // or one that is not there
        const int64_t c = column / per_class;
        return c < kPairClasses ? (column - c * per_class) * kPairClasses + c : INT64_MAX;
    }
    __host__ __device__ int64_t count() const { return (int64_t)kPairClasses * per_class; }
};

static inline int64_t pair_tiles(int64_t n) { return (n + kPairTile - 1) / kPairTile; }
// bytes of the copy of n rows (whole tiles), and columns of a table of n vectors
static inline int64_t pair_packed_bytes(int64_t n, int64_t dim) {
    return pair_tiles(n) * (kPairTile / kPairStrip) * pair_units(dim).pitch * kPairUnit;
}
static inline int64_t pair_columns(int64_t n_vectors) { return pair_tiles(PairColumns(n_vectors).count()) * kPairTile; }

// Whether a launch takes tables of that size.
bool vl_pair_table_fits(int64_t n_queries, int64_t n_vectors, int64_t dim);

// out[r * columns + PairColumns(n_vectors).of(v)] = distance of queries[r] and vectors[v] as bits (columns of no vector hold
// values nobody asks for).  *unordered becomes 1 if a distance may not be a number below VL_MAXFLOAT.
// packed_queries / packed_vectors: room for the copies (pair_packed_bytes of n_queries and of pair_columns), 16-byte aligned.
// Nothing is allocated or waited for.
int vl_launch_pair_table(const float *queries, int64_t n_queries, const float *vectors, int64_t n_vectors, int64_t dim,
                         int metric, uint8_t *packed_queries, uint8_t *packed_vectors, uint32_t *out, int64_t columns,
                         int *unordered, hipStream_t st);
