// Exact k nearest neighbours of a few queries for gfx950.
//
// The tiles of knn.hip pay for 128 queries whatever the batch holds and cut a table into at most 64 strips, so one query
// against 32,768 x 768 entry points ran on 64 of 256 compute units (235 us).  With few queries the pass is bound by
// reading the table once.  Here a wavefront takes 32 vectors at a time against 32 query columns, operands straight
// from memory into registers (nothing is shared that LDS could serve: the table is read once, the queries sit in the
// caches), and as many wavefronts as the chip holds share the table tile by tile.  v_mfma_f32_32x32x2_f32 covers 32
// columns at 64 cycles per 256 bytes of the table and SIMD - 9.8 TB/s over the chip, above what memory delivers - so the
// idle columns of a smaller batch cost nothing.  Same products in the same order as the tiles: same bits.
// Measured (k = 16, one query): 32,768 x 768 25 us + 10 us selection (4.0 TB/s; 235 + 10 us with the tiles), 500,000 x 768
// 474 us (3.2 TB/s; 3,161), 1,000,000 x 96 171 us (1,108).
#include "knn_device.h"
#include "knn_few.h"

namespace {

constexpr int kFewWaves = 2048;     // most wavefronts that share a table: two per SIMD of 256 compute units
constexpr int kSelectThreads = 1024;

// Every wavefront's list of the KK best per query column and half-wave, as in knn_tile_kernel.
template <int KK, bool L2>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void knn_few_kernel(const float *__restrict__ queries, int n_queries, const float *__restrict__ vectors, int64_t n_vectors,
                    int dim, int n_waves, uint64_t *__restrict__ cand, const float *__restrict__ q_norm,
                    const float *__restrict__ v_norm) {
    const int lane = threadIdx.x & (kWave - 1);
    const int half = lane >> 5, l32 = lane & 31;
    // (workgroups of the query groups that take the same vectors are neighbours: the caches serve all but the first)
    const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.y * 4 + threadIdx.x / kWave));
    if (wave >= n_waves) return;
    const int q = (int)blockIdx.x * 32 + l32;
    const int q_row = min(q, n_queries - 1);  // columns past the last query repeat it; nothing of them is kept
    const float *const pb = queries + (int64_t)q_row * dim + 4 * half;
    const float qn = L2 ? q_norm[q_row] : 0.0f;
    uint64_t *const dst = cand + ((int64_t)q_row * (2 * n_waves) + 2 * wave + half) * KK;

    float kd[KK];
    int32_t kid[KK];
#pragma unroll
    for (int i = 0; i < KK; ++i) {
        kd[i] = __builtin_inff();
        kid[i] = VL_MAXINT;
    }
    float bound = __builtin_inff();
    const int64_t tiles = (n_vectors + 31) / 32;
    for (int64_t tile = wave; tile < tiles; tile += n_waves) {
        const int64_t v0 = tile * 32;
        const int64_t row = v0 + l32 < n_vectors ? v0 + l32 : n_vectors - 1;
        floatx16 acc;
        dot_tile<8>(vectors + row * dim + 4 * half, pb, dim, half, acc);
        // accumulator register r of this lane: vector row 8 * (r / 4) + 4 * half + r % 4, query column l32
        float d[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float vn = 0.0f;
            if constexpr (L2) {
                const int64_t v = v0 + 8 * (r >> 2) + 4 * half + (r & 3);
                vn = v_norm[v < n_vectors ? v : n_vectors - 1];
            }
            d[r] = tile_distance<L2>(acc[r], qn, vn);
        }
        const int v_lane = (int)v0 + 4 * half, v_limit = (int)n_vectors;  // ids stay below 2^30
        if (KK == 16 && tiles <= n_waves) {
            // the wavefront's only tile: its 16 values per lane are the list, the smallest first
            uint64_t key[16], least = kPadKey;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int v = v_lane + 8 * (r >> 2) + (r & 3);
                key[r] = v < v_limit && d[r] < __builtin_inff() ? vl_make_key(v, d[r]) : kPadKey;  // as list_insert takes them
                least = key[r] < least ? key[r] : least;
            }
            if (q < n_queries) {
                dst[0] = least;
#pragma unroll
                for (int r = 1; r < 16; ++r) dst[r] = key[r] == least ? key[0] : key[r];
            }
            return;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int v = v_lane + 8 * (r >> 2) + (r & 3);
            const bool good = v < v_limit && !(d[r] > bound) && d[r] < kd[KK - 1];
            if (__ballot(good) == 0) continue;
            if (good) list_insert<KK>(kd, kid, d[r], v);
        }
        const float own = kd[KK - 1];
        bound = fminf(fminf(own, __shfl_xor(own, 32)), bound);
    }
    if (q >= n_queries) return;
#pragma unroll
    for (int i = 0; i < KK; ++i) dst[i] = kid[i] == VL_MAXINT ? kPadKey : vl_make_key(kid[i], kd[i]);
}

// One workgroup per query picks the k best of its lists.  Only the head of a list is known to be its smallest key.
// Sixteen wavefronts take a sixteenth of the lists each; the k-th smallest of their smallest heads bounds the k-th best
// of all, so the keys up to that bound - a few dozen among thousands of lists whose rows come in any order - are collected
// in LDS and ranked against each other.  (Taking the k smallest heads one by one costs k workgroup-wide minima: 20 us
// instead of 9 for k = 16.)  When more keys than the pool holds are that close - the best rows all in a few wavefronts'
// tiles - the heads are taken one by one after all: a key can only be among the k best if its list's head is among the k
// smallest heads.
constexpr int kPool = 1024;

__global__ __launch_bounds__(kSelectThreads) void knn_few_select_kernel(const uint64_t *__restrict__ cand, int n_lists,
                                                                        int len, int k, int32_t *__restrict__ ids_out,
                                                                        float *__restrict__ d_out) {
    constexpr int kWaves = kSelectThreads / kWave, kMost = 16;
    static_assert(2 * kFewWaves <= 4 * kSelectThreads, "four lists per thread cover all of them");
    __shared__ uint64_t smallest_s[kWaves];
    __shared__ uint64_t pool[kPool];
    __shared__ int pool_n;
    __shared__ uint64_t part_key[kWaves * kMost];
    __shared__ int part_list[kWaves * kMost];
    __shared__ int list_s[kMost];
    const int64_t q = blockIdx.x;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1), wave = tid / kWave;
    const uint64_t *base = cand + q * n_lists * len;
    const int first = lane * kWaves + wave;  // lists first, first + 1024, ...: a short table's spread over the wavefronts too
    uint64_t head[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int list = first + kSelectThreads * j;
        head[j] = list < n_lists ? base[(int64_t)list * len] : kPadKey;
    }
    auto smallest_of = [](const uint64_t (&h)[4]) {
        uint64_t m = h[0];
#pragma unroll
        for (int j = 1; j < 4; ++j) m = h[j] < m ? h[j] : m;
        return m;
    };
    const uint64_t mine = smallest_of(head);
    const uint64_t wave_smallest = wave_min_u64(mine);
    if (lane == 0) smallest_s[wave] = wave_smallest;
    if (tid == 0) pool_n = 0;
    __syncthreads();
    uint64_t bound;
    {
        // the one of rank k - 1 (equal ones, which are all empty, are told apart by place)
        const uint64_t x = smallest_s[lane & (kWaves - 1)];
        int rank = 0;
#pragma unroll
        for (int i = 0; i < kWaves; ++i) {
            const uint64_t y = smallest_s[i];
            rank += y < x || (y == x && i < (lane & (kWaves - 1)));
        }
        bound = __shfl((unsigned long long)x, __builtin_ctzll(__ballot(rank == k - 1)));
    }
    if (mine <= bound) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (head[j] > bound || head[j] == kPadKey) continue;
            const uint64_t *list = base + (int64_t)(first + kSelectThreads * j) * len;
            for (int i = 0; i < len; ++i) {
                const uint64_t key = list[i];
                if (key > bound || key == kPadKey) continue;
                const int at = atomicAdd(&pool_n, 1);
                if (at < kPool) pool[at] = key;
            }
        }
    }
    __syncthreads();
    int n_keys = pool_n;
    if (n_keys > kPool) {  // uniform over the workgroup
        for (int i = 0; i < k; ++i) {
            const uint64_t own = smallest_of(head);
            const uint64_t best = wave_min_u64(own);
            if (own == best) {  // keys are unique: one lane, unless no list is left
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (head[j] == best) {
                        part_key[wave * k + i] = best;
                        part_list[wave * k + i] = best == kPadKey ? -1 : first + kSelectThreads * j;
                        head[j] = kPadKey;
                    }
            }
        }
        if (tid < kMost) list_s[tid] = -1;
        __syncthreads();
        if (wave == 0) {
            uint64_t left[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) left[j] = lane + kWave * j < kWaves * k ? part_key[lane + kWave * j] : kPadKey;
            for (int i = 0; i < k; ++i) {
                const uint64_t own = smallest_of(left);
                const uint64_t best = wave_min_u64(own);
                if (best == kPadKey) break;
                if (own == best) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (left[j] == best) {
                            list_s[i] = part_list[lane + kWave * j];
                            left[j] = kPadKey;
                        }
                }
            }
        }
        __syncthreads();
        n_keys = k * len;
        if (tid < n_keys) {
            const int list = list_s[tid / len];
            pool[tid] = list < 0 ? kPadKey : base[(int64_t)list * len + tid % len];
        }
        __syncthreads();
    }
    for (int slot = tid; slot < n_keys || slot < k; slot += kSelectThreads) {
        if (slot >= n_keys) {  // fewer keys than asked for: the rest is empty
            ids_out[q * k + slot] = VL_MAXINT;
            d_out[q * k + slot] = VL_MAXFLOAT;
            continue;
        }
        const uint64_t key = pool[slot];
        int rank = 0;
        for (int i = 0; i < n_keys; ++i) {
            const uint64_t other = pool[i];
            rank += other < key || (other == key && i < slot);
        }
        if (rank < k) {
            const bool real = key != kPadKey;
            ids_out[q * k + rank] = real ? vl_key_id(key) : VL_MAXINT;
            d_out[q * k + rank] = real ? vl_key_dist(key) : VL_MAXFLOAT;
        }
    }
}

int few_waves(int64_t n_vectors) {
    const int64_t tiles = (n_vectors + 31) / 32;
    return (int)(tiles < kFewWaves ? tiles : kFewWaves);
}

}  // namespace

int64_t vl_knn_few_lists(int64_t n_vectors) { return 2 * (int64_t)few_waves(n_vectors); }

int vl_knn_few(const float *queries, int64_t n_queries, const float *vectors, int64_t n_vectors, int64_t dim, int64_t k,
               int list_len, bool l2, const float *q_norm, const float *v_norm, uint64_t *cand, int32_t *ids_out,
               float *dists_out, hipStream_t st) {
    VL_REQUIRE(vl_knn_is_few(n_queries, n_vectors, dim), "too many queries for the few-query kernel");
    const int waves = few_waves(n_vectors);
    const dim3 grid((unsigned)((n_queries + 31) / 32), (unsigned)((waves + 3) / 4));
#define VL_FEW_LAUNCH(KERNEL)                                                                                        \
    hipLaunchKernelGGL(KERNEL, grid, dim3(256), 0, st, queries, (int)n_queries, vectors, n_vectors, (int)dim, waves, \
                       cand, q_norm, v_norm)
#define VL_FEW(KK)                                              \
    do {                                                        \
        if (l2) VL_FEW_LAUNCH((knn_few_kernel<KK, true>));      \
        else VL_FEW_LAUNCH((knn_few_kernel<KK, false>));        \
    } while (0)
    switch (list_len) {
        case 1: VL_FEW(1); break;
        case 4: VL_FEW(4); break;
        case 8: VL_FEW(8); break;
        case 10: VL_FEW(10); break;
        case 12: VL_FEW(12); break;
        default: VL_FEW(16); break;
    }
#undef VL_FEW
#undef VL_FEW_LAUNCH
    VL_LAUNCH_CHECK("knn_few_kernel");
    hipLaunchKernelGGL(knn_few_select_kernel, dim3((unsigned)n_queries), dim3(kSelectThreads), 0, st, cand, 2 * waves,
                       list_len, (int)k, ids_out, dists_out);
    VL_LAUNCH_CHECK("knn_few_select_kernel");
    return VL_OK;
}
