// Device code shared by the exact-kNN kernels: staging of operand tiles into LDS, a lane's list of its best, dot
// products of 32 rows with 32 columns straight from memory.
#pragma once
#include "rowsort.h"

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int KT = 32;          // floats of the reduction dimension per stage
constexpr int CH = KT / 4;      // 16-byte chunks per row and stage
constexpr int TILE = 128 * KT;  // floats of one staged operand tile of 128 rows (16 KB)

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void glb_void;

static __device__ __align__(16) const float kZeroChunk[4] = {0.f, 0.f, 0.f, 0.f};

// A lane's list of the KK best so far: distances ascending with their ids.  A lane meets its
// candidates in ascending id order, so one that ties a kept distance belongs behind it: comparing
// distances alone orders (distance, id) pairs correctly.  The new distance column is a median of
// three per slot; ids follow the same comparisons.
template <int KK>
__device__ __forceinline__ void list_insert(float (&kd)[KK], int32_t (&kid)[KK], float d, int32_t id) {
#pragma unroll
    for (int i = KK - 1; i > 0; --i) {
        const bool before_prev = d < kd[i - 1], before_this = d < kd[i];
        kid[i] = before_prev ? kid[i - 1] : (before_this ? id : kid[i]);
        kd[i] = __builtin_amdgcn_fmed3f(kd[i - 1], d, kd[i]);
    }
    const bool first = d < kd[0];
    kid[0] = first ? id : kid[0];
    kd[0] = first ? d : kd[0];
}

// Chunk c (16 bytes) of tile row r lives in slot r * CH + (c ^ swz(r)): sixteen consecutive
// rows read the same chunk index from sixteen different 16-byte bank groups.
__device__ __forceinline__ int swz(int r) { return (r >> 1) & (CH - 1); }

// Staging: 128 rows x KT floats of an operand go straight from global memory into LDS (no
// registers in between).  A wavefront instruction fills 1 KB = 8 tile rows and lane i writes
// slot i of those rows, so it fetches the chunk that belongs there.  Each lane has four such
// (row, chunk) duties per operand; their source addresses at k = 0 are kept as pointers.
// Rows past `last` repeat row `last` (their results are discarded later).  list: the rows' numbers, or null.
__device__ __forceinline__ void duty_pointers(const float *__restrict__ src, int64_t first, int64_t last, int dim,
                                              int wave, int lane, const float *(&p)[4],
                                              const int32_t *__restrict__ list = nullptr) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 8 * (4 * wave + i) + (lane >> 3);
        const int c = (lane & (CH - 1)) ^ swz(r);
        int64_t row = first + r;
        row = row < last ? row : last;
        if (list) row = list[row];
        p[i] = src + row * dim + 4 * c;
    }
}

// RAGGED: the last stage reaches past `dim`; chunks out there come from a zero chunk.
template <bool RAGGED>
__device__ __forceinline__ void stage_operand(const float *const (&p)[4], int kt, int dim, float *tile, int wave,
                                              int lane) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float *g = p[i] + kt;
        if constexpr (RAGGED) {
            const int r = 8 * (4 * wave + i) + (lane >> 3);
            const int c = (lane & (CH - 1)) ^ swz(r);
            if (kt + 4 * c >= dim) g = kZeroChunk;
        }
        __builtin_amdgcn_global_load_lds((glb_void *)g, (lds_void *)(tile + 8 * (4 * wave + i) * KT), 16, 0, 0);
    }
}


// The distance of a dot product; L2 from the squared lengths of the two rows.
template <bool L2>
__device__ __forceinline__ float tile_distance(float dot, float q_norm, float v_norm) {
    if constexpr (L2) return fmaxf(fmaf(-2.0f, dot, q_norm + v_norm), 0.0f);
    const float d = (1.0f - dot) * 0.5f;
    return d < 0.0f ? 0.0f : (d > 1.0f ? 1.0f : d);
}

// One wavefront: the 32 x 32 dot products of the rows its lanes point at with 32 query rows, operands straight from
// memory.  pa / pb: the row of lane & 31, plus 4 floats for the upper half of the wavefront.  The products
// go through v_mfma_f32_32x32x2_f32 in the order of knn_tile_kernel (elements x, y, z, w of chunk pair after chunk pair),
// so the sums have its bits.  U chunk pairs (U KB of the rows) are on their way while as many are multiplied.
template <int U>
__device__ __forceinline__ void dot_tile(const float *pa, const float *pb, int dim, int half, floatx16 &acc) {
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    const int full = dim >> 3;
    float4 a0[U], b0[U], a1[U], b1[U];
    auto load = [&](float4 (&a)[U], float4 (&b)[U], int c0) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (c0 + u < full) {  // uniform
                a[u] = *reinterpret_cast<const float4 *>(pa + 8 * (c0 + u));
                b[u] = *reinterpret_cast<const float4 *>(pb + 8 * (c0 + u));
            }
    };
    auto step = [&](const float4 &x, const float4 &y) {
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x.x, y.x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x.y, y.y, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x.z, y.z, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x.w, y.w, acc, 0, 0, 0);
    };
    auto multiply = [&](const float4 (&a)[U], const float4 (&b)[U], int c0) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (c0 + u < full) step(a[u], b[u]);
    };
    load(a0, b0, 0);
    for (int c = 0; c < full; c += 2 * U) {
        load(a1, b1, c + U);
        __builtin_amdgcn_sched_barrier(0);  // those loads are on their way before this half's products
        multiply(a0, b0, c);
        if (c + U >= full) break;
        load(a0, b0, c + 2 * U);
        __builtin_amdgcn_sched_barrier(0);
        multiply(a1, b1, c + U);
    }
    if (dim & 7) {  // a last chunk pair of which the rows hold the first half only
        const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
        const float4 a = half ? zero : *reinterpret_cast<const float4 *>(pa + 8 * full);
        const float4 b = half ? zero : *reinterpret_cast<const float4 *>(pb + 8 * full);
        step(a, b);
    }
}
