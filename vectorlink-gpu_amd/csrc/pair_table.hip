// Distances of all pairs of a batch of queries and a table of vectors on the matrix cores, with the bits that the gathered
// distances have (dist_device.h): v_mfma_f32_32x32x2_f32 adds its two products to a sum one after the other with the
// rounding of v_fma_f32 (denormals and infinities included), so the four elements that a chunk adds to a partial sum are two
// instructions, and the 63 additions of the folds are left for the vector unit.  Squared differences (VL_METRIC_L2) are
// no products of the operands; the vector unit forms those from the same tiles.
//
// What bounds it: these products run on the vector unit's multipliers (157 TFLOP/s either way), so the additions of the folds,
// one per partial sum and pair, take their time from them: at most 135 TFLOP/s at 768 columns, 105 at 128.  Measured with what
// packs the operands: 10,000 x 20,011 x 768 2.95 ms (104 TFLOP/s), x 1,536 5.65 (109), 10,000 x 100,000 x 128 3.0 (85), 10,000 x
// 40,000 x 130 1.50 (69), 256 x 4,096 x 128 17 us; squared differences 6,007 x 6,007 x 384 0.69 ms (40; beyond 128 columns that kernel keeps 34 registers in
// scratch memory).  Tried and left out:
// tiles of 128 x 64 and 128 x 128 (half the operands from L2: 3,060 and 3,030 us for the first), three and four stages in
// flight (3,000 to 3,060), the operands of the next unit read ahead (3,010), partial sums one at a time (3,600).
#include "pair_table.h"
#include "dist_device.h"

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void glb_void;


__host__ __device__ constexpr int reversed(int x, int bits) {
    int r = 0;
    for (int i = 0; i < bits; ++i) r |= ((x >> i) & 1) << (bits - 1 - i);
    return r;
}

// Queries and vectors; a wavefront for kPackUnits units of a strip.
constexpr int kPackUnits = 8;
struct PackSide {
    const float *rows;
    int64_t n, strips;
    uint8_t *out;
    bool aligned;
    bool by_class;  // the rows are the columns of a table (PairColumns)
};
__global__ __launch_bounds__(256) void pair_pack_kernel(PackSide first, PackSide second, int dim, PairUnits units) {
    const int lane = threadIdx.x & (kWave - 1);
    const int per_strip = (units.count + kPackUnits - 1) / kPackUnits;
    const int64_t item = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    int64_t strip = item / per_strip;
    const int begin = (int)(item - strip * per_strip) * kPackUnits;
    const bool of_first = strip < first.strips;
    const PackSide side = of_first ? first : second;
    if (!of_first) strip -= first.strips;
    if (strip >= side.strips) return;
    int64_t row = strip * kPairStrip + (lane & 31);
    if (side.by_class) row = PairColumns(side.n).vector_at(row);
    const float *const src = side.rows + (row < side.n ? row : 0) * dim;
    const int half = units.sums / 2, bits = 31 - __builtin_clz(half);
    int u = 0;  // the unit that pair p begins with
    for (int p = 0; p < half && u < begin + kPackUnits; ++p) {
        const int c = (int)(__builtin_bitreverse32((uint32_t)p) >> (32 - bits));
        const int count = pair_units_of(units.nchunks, units.sums, c);
        for (int j = max(0, begin - u); j < count && u + j < begin + kPackUnits; ++j) {
            // lanes 0 .. 31 bring the lower chunk, the others the upper one
            const int at = 4 * (c + (lane >= 32 ? half : 0) + units.sums * j);
            float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
            if (row < side.n && at < dim) {
                if (side.aligned) {
                    x = *reinterpret_cast<const float4 *>(src + at);
                } else {
                    x.x = src[at];
                    if (at + 1 < dim) x.y = src[at + 1];
                    if (at + 2 < dim) x.z = src[at + 2];
                    if (at + 3 < dim) x.w = src[at + 3];
                }
            }
            float2 *const to = reinterpret_cast<float2 *>(side.out + (strip * units.pitch + u + j) * kPairUnit) +
                               2 * (lane & 31) + (lane >> 5);
            to[0] = make_float2(x.x, x.z);
            to[64] = make_float2(x.y, x.w);
        }
        u += count;
    }
}

// x + y, added here and not where the sum is used: an addition put off keeps both sides in registers (2,000 were spilled).
__device__ __forceinline__ floatx16 added_here(const floatx16 &x, const floatx16 &y) {
    floatx16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        float one = x[i] + y[i];
        asm volatile("" : "+v"(one));
        s[i] = one;
    }
    return s;
}

// A workgroup's tile: two strips of queries x two of vectors, 32 x 32 for each of its wavefronts.  LDS holds two stages of units
// of each strip, unit u in place u mod 8.
// It is read with instructions written here: the compiler cannot tell the stage that is read from the one that comes in, and
// waits for the loads on their way before every read (10,000 x 20,011 x 768 3,077 us with the compiler's reads, 2,939 so).
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float2v __attribute__((ext_vector_type(2)));
struct PairTile {
    static constexpr int kStripBytes = 2 * kPairStage * (int)kPairUnit, kBytes = 4 * kStripBytes;
    unsigned char *lds;
    const uint8_t *from;   // the next stage of the strip that this wavefront brings in
    int units, u;          // u: the unit that is read next
    int stage_place;       // where in a strip's LDS that stage goes
    int wave, lane;
    uint32_t q, v;         // LDS addresses of the wavefront's strips of queries and vectors

    __device__ __forceinline__ void bring() {
        unsigned char *const to = lds + wave * kStripBytes + stage_place;
#pragma unroll
        for (int i = 0; i < kPairStage; ++i)
            __builtin_amdgcn_global_load_lds((glb_void *)(from + i * kPairUnit + (uint32_t)(lane * 16)),
                                             (lds_void *)(to + i * kPairUnit), 16, 0, 0);
        from += kPairStage * kPairUnit;
        stage_place ^= kPairStage * (int)kPairUnit;
    }
    // Unit u is in LDS.  At the first unit of a stage all wavefronts meet: the stage has landed, the one before is done
    // with, and the next may come in over it.
    __device__ __forceinline__ void arrive() {
        if (u % kPairStage == 0 && u < units) {  // uniform over the workgroup
            __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
            __syncthreads();
            if (u + kPairStage < units) bring();
        }
    }
    __device__ __forceinline__ uint32_t place() const { return (uint32_t)(u % (2 * kPairStage)) * (uint32_t)kPairUnit; }
};

// Folded sums of the pair of partial sums c, of a lane's 16 pairs of a query and a vector.
template <bool L2>
struct PairSums;

template <>
struct PairSums<false> {
    PairTile t;
    float4v a, b;

    __device__ __forceinline__ void read() {
        t.arrive();
        const uint32_t q = t.q + t.place(), v = t.v + t.place();
        asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)" : "=&v"(a), "=&v"(b) : "v"(q), "v"(v) : "memory");
        ++t.u;
    }
    __device__ __forceinline__ floatx16 of(int c, int nchunks, int sums) {
        floatx16 lower = {}, upper = {};
        if (c >= nchunks) return lower;  // uniform
        read();
        lower = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b.x, lower, 0, 0, 0);
        if (c + sums / 2 >= nchunks) return __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, lower, 0, 0, 0);  // the upper one has no chunk
        upper = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b.z, upper, 0, 0, 0);
        lower = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, lower, 0, 0, 0);
        upper = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b.w, upper, 0, 0, 0);
        for (c += sums; c < nchunks; c += sums) {
            read();
            lower = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b.x, lower, 0, 0, 0);
            if (c + sums / 2 < nchunks) upper = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b.z, upper, 0, 0, 0);
            lower = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, lower, 0, 0, 0);
            if (c + sums / 2 < nchunks) upper = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b.w, upper, 0, 0, 0);
        }
        return added_here(lower, upper);
    }
};

template <>
struct PairSums<true> {
    PairTile t;

    // Elements 0 and 2 (xz), 1 and 3 (yw) of four queries or vectors, the unit's lower chunk or its upper.
    __device__ __forceinline__ void read(uint32_t q, uint32_t v, float2v (&qxz)[4], float2v (&qyw)[4], float2v (&vxz)[4], float2v (&vyw)[4]) {
        asm volatile("ds_read_b64 %0, %16\n\tds_read_b64 %1, %16 offset:16\n\tds_read_b64 %2, %16 offset:32\n\tds_read_b64 %3, %16 offset:48\n\t"
                     "ds_read_b64 %4, %16 offset:512\n\tds_read_b64 %5, %16 offset:528\n\tds_read_b64 %6, %16 offset:544\n\tds_read_b64 %7, %16 offset:560\n\t"
                     "ds_read_b64 %8, %17\n\tds_read_b64 %9, %17 offset:16\n\tds_read_b64 %10, %17 offset:32\n\tds_read_b64 %11, %17 offset:48\n\t"
                     "ds_read_b64 %12, %17 offset:512\n\tds_read_b64 %13, %17 offset:528\n\tds_read_b64 %14, %17 offset:544\n\tds_read_b64 %15, %17 offset:560\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=&v"(qxz[0]), "=&v"(qxz[1]), "=&v"(qxz[2]), "=&v"(qxz[3]), "=&v"(qyw[0]), "=&v"(qyw[1]), "=&v"(qyw[2]), "=&v"(qyw[3]),
                       "=&v"(vxz[0]), "=&v"(vxz[1]), "=&v"(vxz[2]), "=&v"(vxz[3]), "=&v"(vyw[0]), "=&v"(vyw[1]), "=&v"(vyw[2]), "=&v"(vyw[3])
                     : "v"(q), "v"(v) : "memory");
    }
    __device__ __forceinline__ void add(floatx16 &sum, int upper) {
        float2v qxz[4], qyw[4], vxz[4], vyw[4];
        read(t.q + t.place() + 8 * upper + 64 * (t.lane >> 3), t.v + t.place() + 8 * upper + 64 * (t.lane & 7), qxz, qyw, vxz, vyw);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float dx = vxz[c].x - qxz[r].x, dy = vyw[c].x - qyw[r].x;
                const float dz = vxz[c].y - qxz[r].y, dw = vyw[c].y - qyw[r].y;
                float s = sum[4 * r + c];
                s = __builtin_fmaf(dx, dx, s);
                s = __builtin_fmaf(dy, dy, s);
                s = __builtin_fmaf(dz, dz, s);
                s = __builtin_fmaf(dw, dw, s);
                sum[4 * r + c] = s;
            }
    }
    __device__ __forceinline__ floatx16 of(int c, int nchunks, int sums) {
        floatx16 lower = {}, upper = {};
        for (; c < nchunks; c += sums, ++t.u) {
            t.arrive();
            add(lower, 0);
            if (c + sums / 2 < nchunks) add(upper, 1);
        }
        return added_here(lower, upper);
    }
};

// The sum of 2^LEVEL pairs of partial sums, beginning with the one of number FIRST + rest of 2^BITS (rest: the bits of a
// pair's number above kFoldBits, reversed), folded in the order of dist_device.h.
constexpr int kFoldBits = 3;
template <class Sums, int BITS, int LEVEL, int FIRST>
__device__ __forceinline__ floatx16 pair_fold(Sums &s, int nchunks, int rest) {
    if constexpr (LEVEL == 0) {
        return s.of(reversed(FIRST, BITS) + rest, nchunks, 2 << BITS);
    } else {
        const floatx16 lower = pair_fold<Sums, BITS, LEVEL - 1, FIRST>(s, nchunks, rest);
        const floatx16 upper = pair_fold<Sums, BITS, LEVEL - 1, FIRST + (1 << (LEVEL - 1))>(s, nchunks, rest);
        return added_here(lower, upper);
    }
}
// The whole sum.  The code of eight pairs is gone through again and again (written out for all 32 it is four times as long and
// takes the same time).
template <class Sums, int BITS>
__device__ __forceinline__ floatx16 pair_sum(Sums &s, int nchunks) {
    if constexpr (BITS == kFoldBits) {
        return pair_fold<Sums, BITS, kFoldBits, 0>(s, nchunks, 0);
    } else {
        floatx16 one = {}, two = {}, sum = {};
#pragma unroll 1
        for (int g = 0; g < 1 << (BITS - kFoldBits); ++g) {
            const int rest = (int)(__builtin_bitreverse32((uint32_t)g) >> (32 - (BITS - kFoldBits)));
            sum = pair_fold<Sums, BITS, kFoldBits, 0>(s, nchunks, rest);
            if ((g & 1) == 0) {
                one = sum;
            } else {
                sum = added_here(one, sum);
                if ((g & 2) == 0) two = sum;
            }
        }
        if constexpr (BITS == kFoldBits + 2) return added_here(two, sum);
        return sum;
    }
}

template <bool L2, int BITS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(L2 ? 3 : 4)))
void pair_tile_kernel(const uint8_t *__restrict__ packed_queries, int64_t n_queries, const uint8_t *__restrict__ packed_vectors,
                      PairUnits units, int row_tiles, int col_tiles, uint32_t *__restrict__ out,
                      int64_t columns, int *__restrict__ unordered) {
    __shared__ __align__(16) unsigned char lds[PairTile::kBytes];
    // Workgroups are dealt to the 8 XCDs in turn; each takes an eighth of the tiles in the order of eight rows of tiles at
    // a time, column by column, so that what its compute units multiply together stays in its L2.
    int row_tile, col_tile;
    {
        const int64_t total = (int64_t)row_tiles * col_tiles, per = (total + 7) >> 3;
        const int64_t k = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
        if ((int64_t)(blockIdx.x >> 3) >= per || k >= total) return;
        const int64_t band = k / (8 * (int64_t)col_tiles), in = k - band * 8 * col_tiles;
        const int rows = min(8, row_tiles - 8 * (int)band);
        col_tile = (int)(in / rows);
        row_tile = 8 * (int)band + (int)(in - (int64_t)col_tile * rows);
    }
    PairSums<L2> sums;
    PairTile &t = sums.t;
    t.lds = lds;
    t.lane = threadIdx.x & (kWave - 1);
    t.wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    t.units = units.count;
    t.u = 0;
    t.stage_place = 0;
    t.q = (uint32_t)(uintptr_t)(lds_void *)lds + (t.wave >> 1) * PairTile::kStripBytes;
    t.v = (uint32_t)(uintptr_t)(lds_void *)lds + (2 + (t.wave & 1)) * PairTile::kStripBytes;
    if constexpr (!L2) {
        t.q += 16 * t.lane;
        t.v += 16 * t.lane;
    }
    t.from = t.wave < 2 ? packed_queries + (2 * (int64_t)row_tile + t.wave) * units.pitch * kPairUnit
                        : packed_vectors + (2 * (int64_t)col_tile + t.wave - 2) * units.pitch * kPairUnit;
    t.bring();
    const floatx16 sum = pair_sum<PairSums<L2>, BITS>(sums, units.nchunks);

    // (addresses: what the rows have in common in scalar registers, a lane's own part is the same for all of them)
    const int64_t row0 = (2 * (int64_t)row_tile + (t.wave >> 1)) * kPairStrip;
    const int64_t col0 = (2 * (int64_t)col_tile + (t.wave & 1)) * kPairStrip;
    uint32_t *const to = out + row0 * columns + col0;
    const uint32_t row_in = L2 ? 4 * (t.lane >> 3) : 4 * (t.lane >> 5), col_in = L2 ? 4 * (t.lane & 7) : t.lane & 31;
    const uint32_t own = row_in * (uint32_t)columns + col_in;  // below 2^31
    const int rows_left = (int)min((int64_t)kPairStrip, n_queries - row0);
    float odd = 0.0f, most = 0.0f;  // odd: 0, or not a number if one of the sums is none or infinite
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int row = L2 ? i >> 2 : 8 * (i >> 2) + (i & 3), col = L2 ? i & 3 : 0;
        odd = __builtin_fmaf(sum[i], 0.0f, odd);
        const float d = L2 ? sum[i] : __builtin_amdgcn_fmed3f((1.0f - sum[i]) * 0.5f, 0.0f, 1.0f);
        if constexpr (L2) most = fmaxf(most, d);
        if ((int)row_in + row < rows_left) (to + row * columns + col)[own] = __builtin_bit_cast(uint32_t, d);
    }
    // (a strip's rows past the last vector are zeros: nothing odd in them, and a squared distance that is one of a query and the origin)
    if (__ballot(!(odd == 0.0f) || !(most < VL_MAXFLOAT)) && t.lane == 0) *unordered = 1;  // every writer stores the same 1
}

template <bool L2>
void launch_tiles(const uint8_t *q, int64_t n_queries, const uint8_t *v, int64_t n_columns, const PairUnits &units, uint32_t *out,
                  int64_t columns, int *unordered, hipStream_t st) {
    const int row_tiles = (int)pair_tiles(n_queries), col_tiles = (int)pair_tiles(n_columns);
    const unsigned grid = (unsigned)(8 * (((int64_t)row_tiles * col_tiles + 7) / 8));
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, st, q, n_queries, v, units, row_tiles, col_tiles, out,
                           columns, unordered);
    };
    if (units.sums == 16) go(pair_tile_kernel<L2, 3>);
    else if (units.sums == 32) go(pair_tile_kernel<L2, 4>);
    else go(pair_tile_kernel<L2, 5>);
}

int64_t pack_blocks(int64_t n_queries, int64_t n_vectors, int64_t dim) {
    const int64_t strips = pair_tiles(n_queries) * (kPairTile / kPairStrip) + pair_columns(n_vectors) / kPairStrip;
    return (strips * ((pair_units(dim).count + kPackUnits - 1) / kPackUnits) + 3) / 4;
}
}  // namespace

bool vl_pair_table_fits(int64_t n_queries, int64_t n_vectors, int64_t dim) {
    const int64_t n_columns = pair_columns(n_vectors);
    return n_columns < (1 << 26) && pair_tiles(n_queries) * pair_tiles(n_columns) < 4 * kMaxBlocks &&
           pack_blocks(n_queries, n_vectors, dim) < 4 * kMaxBlocks;
}

int vl_launch_pair_table(const float *queries, int64_t n_queries, const float *vectors, int64_t n_vectors, int64_t dim,
                         int metric, uint8_t *packed_queries, uint8_t *packed_vectors, uint32_t *out, int64_t columns,
                         int *unordered, hipStream_t st) {
    const PairUnits units = pair_units(dim);
    const int64_t n_columns = pair_columns(n_vectors);
    auto side = [&](const float *rows, int64_t n, int64_t padded, uint8_t *to, bool by_class) {
        return PackSide{rows, n, padded / kPairStrip, to, dim % 4 == 0 && (uintptr_t)rows % 16 == 0, by_class};
    };
    const PackSide q = side(queries, n_queries, pair_tiles(n_queries) * kPairTile, packed_queries, false);
    const PackSide v = side(vectors, n_vectors, n_columns, packed_vectors, true);
    const int64_t blocks = pack_blocks(n_queries, n_vectors, dim);
    VL_REQUIRE(columns >= n_columns && vl_pair_table_fits(n_queries, n_vectors, dim),
               "a table of %lld x %lld distances is too large for one call", (long long)n_queries, (long long)n_vectors);
    hipLaunchKernelGGL(pair_pack_kernel, dim3((unsigned)blocks), dim3(256), 0, st, q, v, (int)dim, units);
    VL_LAUNCH_CHECK("pair_pack_kernel");
    if (metric == VL_METRIC_L2)
        launch_tiles<true>(packed_queries, n_queries, packed_vectors, n_columns, units, out, columns, unordered, st);
    else
        launch_tiles<false>(packed_queries, n_queries, packed_vectors, n_columns, units, out, columns, unordered, st);
    VL_LAUNCH_CHECK("pair_tile_kernel");
    return VL_OK;
}
