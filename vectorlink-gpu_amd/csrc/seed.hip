// The search queue that a search starts from (ann.py:217-232), in one launch: a row's seeds, their distances, and the queue row
// that Queue.insert (queue.py:37-61) makes of them when nothing is queued yet.  As single steps - two fills, seeds, distances, the
// insert, for dense seeds also the translation of entry points to ids - each of them is some 5 us of work behind 10 to 30 us
// of the host's, and a search of one query waits for all of them (one query at 100,000 x 768 222 us so, 167 in one launch).
#include "dist_device.h"
#include "rowsort.h"

namespace {

struct SeedArgs {
    const float *queries, *vectors;
    const int32_t *seeds;   // [rows, k], or (circulant) the k numbers that are added to a row's own
    const int32_t *names;   // what a seed of `seeds` is called, or null: an id already
    int32_t *q_ids;
    float *q_d;
    int64_t row0, n_vectors, n_names;
    int dim, nchunks, k, cap, P, cw;
    int circulant, l2;
};

template <int CPL, int LPR, int U, RowForm FORM>
__global__ __launch_bounds__(kQueueThreads) void seed_queue_kernel(SeedArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    uint64_t *const keys = reinterpret_cast<uint64_t *>(smem);
    int32_t *const ids = reinterpret_cast<int32_t *>(keys + a.P);
    float *const dists = reinterpret_cast<float *>(ids + a.k);
    __shared__ PlaceScratch ps;
    __shared__ int beyond_s;
    const int64_t row = a.row0 + blockIdx.x;
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    auto real = [&](int32_t id) { return id != VL_MAXINT && id >= 0 && (int64_t)id < a.n_vectors; };
    for (int i = threadIdx.x; i < a.k; i += kQueueThreads) {
        int32_t id;
        if (a.circulant) {
            id = (int32_t)((row + a.seeds[i]) % a.n_vectors);  // utils.py:26-32 (the order is the queue's)
        } else {
            id = a.seeds[row * a.k + i];
            if (a.names) id = id >= 0 && (int64_t)id < a.n_names ? a.names[id] : VL_MAXINT;
        }
        ids[i] = id;
        if (!real(id)) dists[i] = VL_MAXFLOAT;
    }
    if (threadIdx.x == 0) beyond_s = 0;
    __syncthreads();
    const float *const q_row = a.queries + row * a.dim;
    for (int c0 = wave * a.cw; c0 < a.k; c0 += kQueueWaves * a.cw) {
        const bool has = lane < min(a.cw, a.k - c0);
        const int32_t id = has ? ids[c0 + lane] : VL_MAXINT;
        if constexpr (FORM == kRowScalar)
            wave_distances_generic(q_row, a.vectors, a.dim, a.nchunks, id, real(id), dists + c0, nullptr, 0, a.l2 != 0);
        else
            wave_distances<CPL, LPR, U, FORM == kRowUnaligned>(q_row, a.vectors, a.dim, a.nchunks, id, real(id), dists + c0, nullptr,
                                                               0, a.l2 != 0);
    }
    __syncthreads();
    // The row is its seeds, sorted, and empty pairs.  (With a distance beyond VL_MAXFLOAT those come between two seeds: the
    // empty pairs are sorted with them then.)
    for (int i = threadIdx.x; i < a.k; i += kQueueThreads)
        if (!(dists[i] <= VL_MAXFLOAT)) beyond_s = 1;  // every writer stores the same 1
    __syncthreads();
    const int n = beyond_s ? a.cap : a.k;
    int P = 2;
    while (P < n) P <<= 1;
    for (int i = threadIdx.x; i < P; i += kQueueThreads)
        keys[i] = i < a.k ? vl_make_key(ids[i], dists[i]) : i < n ? vl_make_key(VL_MAXINT, VL_MAXFLOAT) : kPadKey;
    block_bitonic_sort(keys, P);
    block_place3(keys, n, a.cap, a.q_ids + row * a.cap, a.q_d + row * a.cap, &ps, nullptr, 0, nullptr, nullptr, a.cap - n);
}

template <int CPL, int LPR, int U, RowForm FORM>
hipError_t launch_seeds(const SeedArgs &a, int64_t rows, size_t smem, hipStream_t st) {
    const hipError_t e = vl_allow_lds(seed_queue_kernel<CPL, LPR, U, FORM>, smem);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((seed_queue_kernel<CPL, LPR, U, FORM>), dim3((unsigned)rows), dim3(kQueueThreads), smem, st, a);
    return hipSuccess;
}
template <int CPL, int LPR, int U>
hipError_t launch_seeds(const SeedArgs &a, bool aligned, int64_t rows, size_t smem, hipStream_t st) {
    return aligned ? launch_seeds<CPL, LPR, U, kRowAligned>(a, rows, smem, st) : launch_seeds<CPL, LPR, U, kRowUnaligned>(a, rows, smem, st);
}
// (the shapes of dist.hip)
hipError_t launch_by_length(const SeedArgs &a, bool aligned, int64_t rows, size_t smem, hipStream_t st) {
    const int c = a.nchunks;
    if (c > 512 || (!aligned && a.dim < 4)) return launch_seeds<1, 64, 1, kRowScalar>(a, rows, smem, st);
    if (c <= 16) return launch_seeds<1, 16, 8>(a, aligned, rows, smem, st);
    if (c <= 32) return launch_seeds<2, 16, 4>(a, aligned, rows, smem, st);
    if (c <= 64) return launch_seeds<1, 64, 8>(a, aligned, rows, smem, st);
    if (c <= 96) return launch_seeds<3, 32, 4>(a, aligned, rows, smem, st);
    if (c <= 128) return launch_seeds<2, 64, 8>(a, aligned, rows, smem, st);
    if (c <= 192) return launch_seeds<3, 64, 4>(a, aligned, rows, smem, st);
    if (c <= 256) return launch_seeds<4, 64, 4>(a, aligned, rows, smem, st);
    if (c <= 320) return launch_seeds<5, 64, 2>(a, aligned, rows, smem, st);
    if (c <= 384) return launch_seeds<6, 64, 2>(a, aligned, rows, smem, st);
    if (c <= 448) return launch_seeds<7, 64, 2>(a, aligned, rows, smem, st);
    return launch_seeds<8, 64, 2>(a, aligned, rows, smem, st);
}

}  // namespace

VL_EXPORT int vl_seed_queue(const float *queries, int64_t n_rows, const float *vectors, int64_t n_vectors, int64_t dim, int metric,
                            const int32_t *seeds, int64_t n_seeds, int circulant, const int32_t *names, int64_t n_names,
                            int32_t *q_ids, float *q_dists, int64_t capacity, int64_t length, void *stream) {
    VL_REQUIRE(n_rows >= 0 && n_seeds >= 0 && n_names >= 0 && length >= 0, "negative size");
    VL_REQUIRE(n_vectors > 0 && n_vectors <= VL_MAXINT && dim >= 1 && dim <= (1 << 24), "bad sizes");
    VL_REQUIRE(metric == VL_METRIC_COSINE || metric == VL_METRIC_L2, "unknown metric %d", metric);
    VL_REQUIRE(length + n_seeds <= capacity, "%lld seeds do not fit behind the %lld slots of a queue of %lld", (long long)n_seeds,
               (long long)length, (long long)capacity);
    VL_REQUIRE(capacity <= kMaxRowSlots, "row of %lld slots exceeds the %d that fit the LDS sort", (long long)capacity, kMaxRowSlots);
    VL_REQUIRE(!circulant || n_rows <= (1ll << 31) - (1ll << 24), "row index too large for int32 seeds");
    if (n_rows == 0 || capacity == 0) return VL_OK;
    VL_REQUIRE(queries && vectors && (seeds || n_seeds == 0) && q_ids && q_dists, "null pointer");
    SeedArgs a;
    a.queries = queries; a.vectors = vectors; a.seeds = seeds; a.names = names; a.n_names = n_names;
    a.q_ids = q_ids; a.q_d = q_dists; a.n_vectors = n_vectors; a.dim = (int)dim; a.nchunks = (int)((dim + 3) / 4);
    a.k = (int)n_seeds; a.cap = (int)capacity; a.circulant = circulant != 0; a.l2 = metric == VL_METRIC_L2;
    a.P = vl_next_pow2(capacity < 2 ? 2 : capacity);
    // a row's seeds are spread over the four wavefronts
    a.cw = (int)((n_seeds + kQueueWaves - 1) / kQueueWaves);
    a.cw = a.cw < 1 ? 1 : a.cw > kWave ? kWave : a.cw;
    const bool aligned = dim % 4 == 0 && ((uintptr_t)queries | (uintptr_t)vectors) % 16 == 0;
    const size_t smem = (size_t)a.P * 8 + (size_t)n_seeds * 8;
    for (a.row0 = 0; a.row0 < n_rows; a.row0 += kMaxBlocks) {
        const int64_t rows = n_rows - a.row0 < kMaxBlocks ? n_rows - a.row0 : kMaxBlocks;
        VL_HIP(launch_by_length(a, aligned, rows, smem, (hipStream_t)stream));
    }
    VL_LAUNCH_CHECK("seed_queue_kernel");
    return VL_OK;
}
