// The beam-search loop of closest_vectors (vectorlink_gpu/ann.py:38-93) for
// gfx950.
//
// The reference runs ~50 torch ops / Numba launches and at least two blocking
// host round trips per iteration.  Here an iteration has two phases per query
// row:
//   expand  pop the visit-queue heads, gather their neighbour lists, evaluate
//           the candidate distances (dist_device.h);
//   merge   insert the candidates into the search queue (Queue.insert,
//           queue.py:37-61), record the visited ids (add_new_to_seen_,
//           utils.py:61-82) and refill the visit queue with the candidates
//           not yet visited.
// By default both phases of a row run in one workgroup of ONE launch
// (beam_step_kernel); the two-launch form (expand kernel of dist.hip, then a
// merge kernel) is kept behind a flag.  Batch-wide state (first free
// visited-list column, "any row changed") lives in a device control block;
// the host only reads the changed flag every speculative_readahead
// iterations, the cadence at which the reference tests for progress
// (ann.py:68,90-91).
#include "beam_kernels.h"
#include "beam_table.h"
#include "pair_table.h"
#include <stddef.h>
#include <stdlib.h>
#include <algorithm>
#include <atomic>
#include <mutex>

int vl_launch_expand(const float *queries, int64_t n_rows, const float *vectors, int64_t n_vectors,
                     int64_t dim, const int32_t *ids, const int32_t *visit, int64_t n_visit,
                     const int32_t *beams, int64_t n_nodes, int64_t width, int64_t m,
                     int32_t *idx_out, float *dist_out, BeamCtrl *ctrl, int iter, int readahead,
                     int seen_cols, int64_t visit_stride, int count_evals, uint64_t *memo, int memo_slots,
                     int metric, hipStream_t st);

int vl_launch_sketch_queries(const float *queries, int64_t n_rows, int64_t dim, uint8_t *out_rows, hipStream_t st);

namespace {

// Optional per-kernel timing of the loop (off by default): HIP events around
// every expand and merge launch on the caller's stream, summed per call.
struct BeamProfile {
    int enabled = 0;
    double expand_ms = 0, merge_ms = 0;
    int64_t expand_launches = 0, merge_launches = 0, evals = 0, rows = 0, iterations = 0, wanted = 0, sketched = 0;
};
// A call sums into a BeamProfile of its own and adds it here once, under the mutex, when
// it returns, so calls on different host threads do not tear each other's sums.  (The
// library's other mutable state: the launch counter below, the page of report slots in
// beam_report.h, the thread-local error text.)
BeamProfile g_prof;
std::mutex g_prof_mutex;
std::atomic<int64_t> g_step_launches{0};  // vl_beam_launches

// HIP events of one profiled call; destroyed on every way out of the call.
struct EventSet {
    hipEvent_t ev[3 * 64];
    int n = 0;
    int create(int count) {
        for (; n < count; ++n) VL_HIP(hipEventCreate(&ev[n]));
        return VL_OK;
    }
    ~EventSet() {
        for (int i = 0; i < n; ++i) (void)hipEventDestroy(ev[i]);
    }
};

// What beam_report.h asks of the HIP runtime, for the stream of a call.
struct StreamOfCall {
    hipStream_t st;
    static void *pinned(size_t bytes) {
        void *p = nullptr;
        if (hipHostMalloc(&p, bytes, hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent) == hipSuccess) return p;
        (void)hipGetLastError();
        return nullptr;
    }
    int state() const {
        const hipError_t e = hipStreamQuery(st);
        return e == hipSuccess ? 0 : (e == hipErrorNotReady ? 1 : -1 - (int)e);
    }
    bool drain() const { return hipStreamSynchronize(st) == hipSuccess; }
};

__device__ inline bool sorted_contains(const int32_t *a, int n, int32_t v) {
    int lo = 0, hi = n;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (a[mid] < v) lo = mid + 1;
        else hi = mid;
    }
    return lo < n && a[lo] == v;
}
__device__ inline int lower_bound(const int32_t *a, int n, int32_t v) {
    int lo = 0, hi = n;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (a[mid] < v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

constexpr uint64_t kMemoEmpty = (uint64_t)(uint32_t)VL_MAXINT;  // id VL_MAXINT, which no probe asks for
__global__ void beam_memo_clear_kernel(uint64_t *memo, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) memo[i] = kMemoEmpty;
}

// memo: the cache, cleared here as well, or null (a launch of its own is some 10 us to one query).  row_word: what every row starts with in its word of the memo_rate array (StepArgs); sketch_rows: how many rows
// that makes users of the sketch.
__global__ __launch_bounds__(kQueueThreads) void beam_init_kernel(BeamCtrl *ctrl, int64_t n_rows, const int32_t *q_ids,
                                                                 const float *q_d, int cap, int head, int32_t *v_ids,
                                                                 float *v_d, int VL, int32_t *seen_count,
                                                                 int32_t *row_quiet, int32_t *memo_rate, int row_word,
                                                                 int sketch_rows, uint64_t *memo, int64_t memo_slots) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (memo)
        for (int64_t i = t; i < memo_slots; i += (int64_t)gridDim.x * blockDim.x) memo[i] = kMemoEmpty;
    if (t == 0) {
        ctrl->stop = 0;
        ctrl->ended_after = 0;
        ctrl->first[0] = ctrl->first[1] = ctrl->first[2] = 0;
        ctrl->sketch_rows = sketch_rows;
        ctrl->error = 0;
        ctrl->refused_at = 0;
        ctrl->unordered = 0;
    }
    if (t < 64) ctrl->changed[t] = 0;
    if (t < kBeamStripes) {
        ctrl->evals[t] = 0;
        ctrl->wanted[t] = 0;
        ctrl->sketched[t] = 0;
    }
    if (t < n_rows) {
        seen_count[t] = 0;
        row_quiet[t] = 0;
        memo_rate[t] = row_word;
    }
    if (t < n_rows * VL) {  // Queue.initialize_from_queue, queue.py:30-35
        int64_t r = t / VL;
        int i = (int)(t % VL);
        v_ids[t] = i < head ? q_ids[r * cap + i] : VL_MAXINT;
        v_d[t] = i < head ? q_d[r * cap + i] : VL_MAXFLOAT;
    }
}

__global__ __launch_bounds__(kQueueThreads) void beam_merge_kernel(MergeArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int Pmax = a.Ps > a.Pv ? a.Ps : a.Pv;
    uint64_t *keys = reinterpret_cast<uint64_t *>(smem);
    int32_t *before = reinterpret_cast<int32_t *>(keys + Pmax);
    int32_t *seen_a = before + a.L;
    int32_t *seen_b = seen_a + a.E;
    int32_t *exl = seen_b + a.E;
    __shared__ PlaceScratch ps;
    __shared__ int n_ex_s;
    __shared__ int32_t newv[kMaxVisit];
    __shared__ int n_new_s;

    BeamCtrl *c = a.ctrl;
    if (c->stop) return;
    const int t = a.iter;
    const int64_t row = blockIdx.x;
    int cnt = a.seen_count[row];
    int *first_next = &c->first[(t + 1) % 3];
    if (t >= 2 && c->first[(t - 1) % 3] >= a.E) {
        // the visit queue is no longer fed: every candidate of this iteration is
        // empty and no queue changes; keep the running maximum current
        if (threadIdx.x == 0) atomicMax(first_next, cnt);
        return;
    }
    const int first = c->first[t % 3];
    const bool seen_full = first >= a.E;  // add_new_to_seen_ returns None now (utils.py:68-69)
    const bool checking = (t % a.readahead) == 0;

    // ---- search_queue.insert(candidates, exclude) : ann.py:75-80 -----------
    if (threadIdx.x == 0) n_ex_s = a.excl ? a.excl_cols : 0;
    __syncthreads();
    if (a.excl) {
        const int32_t *ex = a.excl + row * a.excl_cols;
        for (int i = threadIdx.x; i < a.excl_cols; i += blockDim.x) {
            int32_t e = ex[i];
            exl[i] = e;
            if (e == VL_MAXINT) atomicMin(&n_ex_s, i);
        }
    }
    int32_t *qi = a.q_ids + row * a.cap;
    float *qd = a.q_d + row * a.cap;
    const int32_t *ci = a.cand_ids + row * a.m;
    const float *cd = a.cand_d + row * a.m;
    for (int i = threadIdx.x; i < a.L; i += blockDim.x) before[i] = qi[i];
    __syncthreads();
    const int n_ex = n_ex_s;
    for (int i = threadIdx.x; i < a.Ps; i += blockDim.x) {
        uint64_t k = kPadKey;
        if (i < a.cap) {
            int32_t id;
            float d;
            if (i >= a.L && i < a.L + a.m) {
                id = ci[i - a.L];
                d = cd[i - a.L];
                bool hit = false;
                for (int e = 0; e < n_ex; ++e) hit |= (exl[e] == id);
                if (hit) {
                    id = VL_MAXINT;
                    d = VL_MAXFLOAT;
                }
            } else {
                id = qi[i];
                d = qd[i];
            }
            k = vl_make_key(id, d);
        }
        keys[i] = k;
    }
    block_bitonic_sort(keys, a.Ps);
    block_place3(keys, a.cap, a.cap, qi, qd, &ps, before, a.L, nullptr,
                 checking ? &c->changed[(t / a.readahead) & 63] : nullptr);

    if (seen_full) {
        if (threadIdx.x == 0) atomicMax(first_next, cnt);
        return;
    }

    // ---- add_new_to_seen_(seen, visited) : utils.py:61-82 -------------------
    // The row is kept sorted, duplicate free and packed at the front, which is
    // what sort + dedup + sort leaves; `cnt` ids are in use.
    int32_t *srow = a.seen + row * a.E;
    const int32_t *vrow_i = a.v_ids + row * a.VL;
    const float *vrow_d = a.v_d + row * a.VL;
    for (int i = threadIdx.x; i < cnt; i += blockDim.x) seen_a[i] = srow[i];
    if (threadIdx.x == 0) n_new_s = 0;
    __syncthreads();
    const int n_add = min(min(a.E - first, a.Vt), a.E - cnt);  // utils.py:73-75 (cnt <= first: rows are packed)
    if (threadIdx.x < kWave) {
        const int j = threadIdx.x;
        int32_t x = j < n_add ? vrow_i[j] : VL_MAXINT;
        bool valid = j < n_add && x != VL_MAXINT && !sorted_contains(seen_a, cnt, x);
        for (int i = 0; i < j && valid; ++i)
            if (vrow_i[i] == x) valid = false;
        uint64_t vm = __ballot(valid);
        // ascending rank among the valid new ids
        int rank = 0;
        for (int i = 0; i < n_add; ++i) {
            int32_t y = vrow_i[i];
            if (((vm >> i) & 1) && y < x) ++rank;
        }
        if (valid) newv[rank] = x;
        if (j == 0) n_new_s = __popcll(vm);
    }
    __syncthreads();
    const int n_new = n_new_s;
    for (int p = threadIdx.x; p < cnt; p += blockDim.x) {
        int32_t v = seen_a[p];
        int shift = 0;
        for (int i = 0; i < n_new; ++i) shift += newv[i] < v;
        seen_b[p + shift] = v;
    }
    if (threadIdx.x < n_new) seen_b[lower_bound(seen_a, cnt, newv[threadIdx.x]) + threadIdx.x] = newv[threadIdx.x];
    __syncthreads();
    cnt += n_new;
    for (int i = threadIdx.x; i < cnt; i += blockDim.x) srow[i] = seen_b[i];
    if (threadIdx.x == 0) {
        a.seen_count[row] = cnt;
        atomicMax(first_next, cnt);
    }

    // ---- visit_queue.insert(candidates, exclude=seen) : ann.py:85-88 --------
    // slots [0, Vt) were popped at the start of this iteration (queue.py:87-95)
    for (int i = threadIdx.x; i < a.Pv; i += blockDim.x) {
        uint64_t k = kPadKey;
        if (i < a.VL + a.m) {
            int32_t id = VL_MAXINT;
            float d = VL_MAXFLOAT;
            if (i >= a.VL) {
                id = ci[i - a.VL];
                d = cd[i - a.VL];
                if (sorted_contains(seen_b, cnt, id)) {
                    id = VL_MAXINT;
                    d = VL_MAXFLOAT;
                }
            } else if (i >= a.Vt) {
                id = vrow_i[i];
                d = vrow_d[i];
            }
            k = vl_make_key(id, d);
        }
        keys[i] = k;
    }
    block_bitonic_sort(keys, a.Pv);
    block_place3(keys, a.VL + a.m, a.VL, a.v_ids + row * a.VL, a.v_d + row * a.VL, &ps, nullptr, 0, nullptr,
                 nullptr);
}

// ---- merge, second form ------------------------------------------------------
// Same result as beam_merge_kernel on [0, length) of the search queue and on the
// visit queue, for queues in the state Queue.insert leaves them (ordered by
// (distance, id), distinct ids) and ids that always carry the same distance -
// both hold for everything closest_vectors is handed by this package.  Instead
// of two full-row sorts, the candidates are sorted once; what is already queued
// (or excluded, or visited) is filtered out with binary searches; the few
// survivors are merged into each sorted queue by rank.
__device__ inline int key_lower_bound(const uint64_t *a, int n, uint64_t k) {
    int lo = 0, hi = n;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (a[mid] < k) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// Order-preserving compaction of src[0:n) by predicate into dst; returns the
// kept count (uniform).  wave_cnt: kQueueWaves ints of LDS.
template <class Pred>
__device__ inline int block_compact(const uint64_t *src, int n, uint64_t *dst, Pred keep, int *wave_cnt) {
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    int run = 0;
    for (int base = 0; base < n; base += blockDim.x) {
        int i = base + threadIdx.x;
        bool k = i < n && keep(i);
        uint64_t b = __ballot(k);
        if (lane == 0) wave_cnt[wave] = __popcll(b);
        __syncthreads();
        if (k) {
            int dest = run + __popcll(b & ((1ull << lane) - 1));
            for (int w = 0; w < wave; ++w) dest += wave_cnt[w];
            dst[dest] = src[i];
        }
        for (int w = 0; w < (int)(blockDim.x / kWave); ++w) run += wave_cnt[w];
        __syncthreads();
    }
    return run;
}

// Smallest value over the workgroup of each thread's `mine` (0xFFFFFFFF = none).
// red: 2 * kQueueWaves words of LDS, used alternately so one barrier per call suffices.
__device__ inline uint32_t block_min_u32(uint32_t mine, uint32_t *red, int round) {
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int nw = blockDim.x / kWave;
    mine = wave_min_u32(mine);
    uint32_t *slot = red + (round & 1) * kQueueWaves;
    if (lane == 0) slot[wave] = mine;
    __syncthreads();
    uint32_t m = slot[0];
    for (int w = 1; w < nw; ++w) m = slot[w] < m ? slot[w] : m;
    return m;
}

// The two-launch form's merge of one row; the candidates come from the expand kernel through memory.
template <int THREADS>
__device__ __forceinline__ void merge_row(const MergeArgs &a, unsigned char *smem) {
    const int Pc = a.Pc;
    uint64_t *raw = reinterpret_cast<uint64_t *>(smem);  // candidate keys as they arrive
    uint64_t *uk = raw + Pc;                             // the candidates that can matter, then sorted
    uint64_t *cc = raw;                                  // filtered for one merge (raw is no longer needed by then)
    uint64_t *qa = uk + Pc;                              // search queue [0, L)
    uint64_t *va = qa + a.L;                             // visit queue [Vt, VL)
    int32_t *seen_a = reinterpret_cast<int32_t *>(va + a.VL);
    int32_t *seen_b = seen_a + a.E;
    int32_t *exl = seen_b + a.E;
    uint8_t *fl = reinterpret_cast<uint8_t *>(exl + a.excl_cols);  // per candidate: bit0 wanted, bit1 rest
    __shared__ int wave_cnt[kQueueWaves];
    __shared__ uint64_t red[2 * kQueueWaves];
    __shared__ int32_t newv[kMaxVisit];  // the ids the merge adds to the visited list
    __shared__ int n_ex_s;               // exclusion ids before the row's first empty one
    __shared__ int n_new_s;

    BeamCtrl *c = a.ctrl;
    const int t = a.iter;
    const int64_t row = blockIdx.x;
    const int lane = threadIdx.x & (kWave - 1);
    int32_t *qi = a.q_ids + row * a.cap;
    float *qd = a.q_d + row * a.cap;
    int32_t *vi = a.v_ids + row * a.VL;
    float *vd = a.v_d + row * a.VL;
    const int32_t *ci = a.cand_ids + row * a.m;
    const float *cd = a.cand_d + row * a.m;
    const int nva = a.VL - a.Vt;
    int *first_next = &c->first[(t + 1) % 3];

    const int stop = c->stop;
    const int first_prev = c->first[(t - 1) % 3];
    const int first = c->first[t % 3];
    int cnt = a.seen_count[row];
    // the ids popped at the start of this iteration (queue.py:87-95), before the row is rewritten
    int32_t popped = VL_MAXINT;
    {
        // the visited list's fill is at most Vt ids per earlier iteration, so the row can be
        // fetched without first waiting for the exact count
        const int seen_bound = min(a.E, a.Vt * (t - 1));
        for (int i = threadIdx.x; i < a.m; i += blockDim.x) raw[i] = vl_make_key(ci[i], cd[i]);
        for (int i = threadIdx.x; i < a.L; i += blockDim.x) qa[i] = vl_make_key(qi[i], qd[i]);
        for (int i = threadIdx.x; i < nva; i += blockDim.x) va[i] = vl_make_key(vi[a.Vt + i], vd[a.Vt + i]);
        {
            const int32_t *srow = a.seen + row * a.E;
            for (int i = threadIdx.x; i < seen_bound; i += blockDim.x) seen_a[i] = srow[i];
        }
        if (threadIdx.x < kWave && (int)threadIdx.x < a.Vt) popped = vi[threadIdx.x];
        if (threadIdx.x == 0) {
            n_ex_s = a.excl ? a.excl_cols : 0;
            n_new_s = 0;
        }
        __syncthreads();
        if (a.excl) {
            const int32_t *ex = a.excl + row * a.excl_cols;
            for (int i = threadIdx.x; i < a.excl_cols; i += blockDim.x) {
                int32_t e = ex[i];
                exl[i] = e;
                if (e == VL_MAXINT) atomicMin(&n_ex_s, i);
            }
        }
    }
    if (stop) return;
    if (!beam_row_state_ok(c, cnt, min(a.E, a.Vt * (t - 1)), threadIdx.x == 0)) return;
    if (t >= 2 && first_prev >= a.E) {
        // the visit queue is no longer fed: every candidate of this iteration is empty
        if (threadIdx.x == 0) raise_running_max(first_next, cnt, min(a.E, a.Vt * t));
        return;
    }
    const bool seen_full = first >= a.E;
    const bool checking = (t % a.readahead) == 0;
    __syncthreads();
    const int n_ex = n_ex_s;

    // ---- add_new_to_seen_ : utils.py:61-82 (does not depend on the candidates) ------
    if (!seen_full) {
        const int n_add = min(min(a.E - first, a.Vt), a.E - cnt);  // cnt <= first: rows are packed
        if (threadIdx.x < kWave) {
            const int j = threadIdx.x;
            int32_t x = j < n_add ? popped : VL_MAXINT;
            bool valid = j < n_add && x != VL_MAXINT && !sorted_contains(seen_a, cnt, x);
            for (int i = 0; i < n_add; ++i) {
                int32_t y = __shfl(popped, i);
                if (i < j && y == x) valid = false;
            }
            uint64_t vm = __ballot(valid);
            int rank = 0;
            for (int i = 0; i < n_add; ++i) {
                int32_t y = __shfl(popped, i);
                if (((vm >> i) & 1) && y < x) ++rank;
            }
            if (valid) newv[rank] = x;
            if (j == 0) n_new_s = __popcll(vm);
        }
        __syncthreads();
        const int n_new = n_new_s;
        for (int p = threadIdx.x; p < cnt; p += blockDim.x) {
            int32_t v = seen_a[p];
            int shift = 0;
            for (int i = 0; i < n_new; ++i) shift += newv[i] < v;
            seen_b[p + shift] = v;
        }
        if ((int)threadIdx.x < n_new)
            seen_b[lower_bound(seen_a, cnt, newv[threadIdx.x]) + threadIdx.x] = newv[threadIdx.x];
        __syncthreads();
        cnt += n_new;
        if (n_new) {
            int32_t *srow = a.seen + row * a.E;
            for (int i = threadIdx.x; i < cnt; i += blockDim.x) srow[i] = seen_b[i];
        }
        if (threadIdx.x == 0 && n_new) a.seen_count[row] = cnt;
    }
    if (threadIdx.x == 0) raise_running_max(first_next, cnt, min(a.E, a.Vt * t));

    // ---- which candidates can matter at all -------------------------------------------
    // search queue: only keys below its last slot can enter.  visit queue (VL slots, Vt of
    // them just freed): every unvisited key below its last live slot, plus the Vt best
    // distinct unvisited keys above it.  Everything else is dropped before the sort.  What is
    // chosen here may be a superset - the merges below are exact and cut by rank - so the keys
    // above the visit queue's last slot ("rest") are looked up in the visited list only when
    // they come up as one of the smallest.
    const uint64_t ws = qa[a.L - 1];
    const uint64_t wv = nva > 0 ? va[nva - 1] : 0ull;
    for (int i = threadIdx.x; i < a.m; i += blockDim.x) {
        uint64_t k = raw[i];
        int32_t id = vl_key_id(k);
        uint8_t f = 0;
        if (id != VL_MAXINT) {
            if (k < ws) f |= 1;
            if (!seen_full && k != wv) {  // k == wv is the visit queue's own last slot again
                bool unseen = !sorted_contains(seen_b, cnt, id);
                if (unseen) f |= (k < wv) ? 1 : 2;
            }
        }
        fl[i] = f;
    }
    // The Vt smallest distinct keys among the "rest" candidates are found by their distances alone (the high
    // word of a key): Vt rounds of a workgroup-wide minimum over 32-bit words give the Vt smallest distinct
    // distances, and every "rest" candidate at or below the last of them is taken - the same candidates, plus
    // others of equal distance when there are ties, which the merges below cut by rank.
    uint32_t sel_max = 0u;  // largest selected distance word among the "rest" candidates
    bool any_rest = false;
    if (!seen_full) {
        uint32_t *red32 = reinterpret_cast<uint32_t *>(red);
        uint32_t last = 0u;
        for (int r = 0; r < a.Vt; ++r) {
            uint32_t mine = 0xFFFFFFFFu;
            for (int i = threadIdx.x; i < a.m; i += blockDim.x) {
                const uint32_t k = (uint32_t)(raw[i] >> 32);
                if ((fl[i] & 2) && (r == 0 || k > last) && k < mine) mine = k;
            }
            const uint32_t mn = block_min_u32(mine, red32, r);
            if (mn == 0xFFFFFFFFu) break;
            last = mn;
            sel_max = mn;
            any_rest = true;
        }
    }
    __syncthreads();
    auto wanted = [&](int i) -> bool {
        uint8_t f = fl[i];
        return (f & 1) || (any_rest && (f & 2) && (uint32_t)(raw[i] >> 32) <= sel_max);
    };
    const int n_u = block_compact(raw, a.m, uk, wanted, wave_cnt);
    int Pu = 2;
    while (Pu < n_u) Pu <<= 1;
    for (int i = n_u + threadIdx.x; i < Pu; i += blockDim.x) uk[i] = kPadKey;
    block_bitonic_sort(uk, Pu);

    // ---- search_queue.insert : ann.py:75-80 -------------------------------------------
    auto keep_search = [&](int i) -> bool {
        uint64_t k = uk[i];
        int32_t id = vl_key_id(k);
        if (i > 0 && id == vl_key_id(uk[i - 1])) return false;   // neighbouring duplicate (kernels.py:314-349)
        if (!(k < ws)) return false;
        for (int e = 0; e < n_ex; ++e)
            if (exl[e] == id) return false;                      // queue.py:52-53
        int p = key_lower_bound(qa, a.L, k);
        return !(p < a.L && qa[p] == k);                         // already queued
    };
    const int n_s = block_compact(uk, n_u, cc, keep_search, wave_cnt);
    bool diff = false;
    if (n_s) {
        for (int i = threadIdx.x; i < a.L; i += blockDim.x) {
            uint64_t k = qa[i];
            int r = i + key_lower_bound(cc, n_s, k);
            if (r != i && r < a.L) {
                qi[r] = vl_key_id(k);
                qd[r] = vl_key_dist(k);
            }
        }
        for (int j = threadIdx.x; j < n_s; j += blockDim.x) {
            uint64_t k = cc[j];
            int r = j + key_lower_bound(qa, a.L, k);
            if (r < a.L) {
                qi[r] = vl_key_id(k);
                qd[r] = vl_key_dist(k);
                diff = true;  // a new id inside the first L slots: the row changed (queue.py:57-59)
            }
        }
    }
    int *flag = &c->changed[(t / a.readahead) & 63];  // every writer stores the same 1: no atomic needed
    if (checking && __ballot(diff) && lane == 0) {
        if (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
            __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (seen_full) return;
    __syncthreads();  // cc is reused below

    // ---- visit_queue.insert(candidates, exclude=seen) : ann.py:85-88 --------------------
    auto keep_visit = [&](int i) -> bool {
        uint64_t k = uk[i];
        int32_t id = vl_key_id(k);
        if (i > 0 && id == vl_key_id(uk[i - 1])) return false;
        if (sorted_contains(seen_b, cnt, id)) return false;                      // kernels.py:471-488
        int p = key_lower_bound(va, nva, k);
        return !(p < nva && va[p] == k);
    };
    const int n_v = block_compact(uk, n_u, cc, keep_visit, wave_cnt);
    for (int i = threadIdx.x; i < nva; i += blockDim.x) {
        uint64_t k = va[i];
        int r = i + key_lower_bound(cc, n_v, k);
        if (r < a.VL) {
            vi[r] = vl_key_id(k);
            vd[r] = vl_key_dist(k);
        }
    }
    for (int j = threadIdx.x; j < n_v; j += blockDim.x) {
        uint64_t k = cc[j];
        int r = j + key_lower_bound(va, nva, k);
        if (r < a.VL) {
            vi[r] = vl_key_id(k);
            vd[r] = vl_key_dist(k);
        }
    }
    for (int r = nva + n_v + threadIdx.x; r < a.VL; r += blockDim.x) {  // the popped slots end up here, empty
        vi[r] = VL_MAXINT;
        vd[r] = VL_MAXFLOAT;
    }
}

template <int THREADS>
__global__ __launch_bounds__(THREADS) void beam_merge2_kernel(MergeArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    merge_row<THREADS>(a, smem);
}

// VL_DIST_VARIANT (experiments only): 1 = two rows per load for rows of up to 512 bytes (32 lanes each) and
// one row per load for rows of up to 1536 bytes, the shapes used before lane groups of 16 / 32 took them over.
int dist_variant() {
    static const int v = [] {
        const char *e = getenv("VL_DIST_VARIANT");
        return e ? atoi(e) : 0;
    }();
    return v;
}

// The numbers after `false` are the sketch's lane shape for rows of that size (chunks per lane, lanes per row,
// loads in flight), the wavefronts per SIMD asked for, the whole rows in flight in the sketch kernel (it fetches
// few of them, so fewer in flight cost nothing and leave registers for another wavefront: 0.40 -> 0.36 ms per
// launch at 384 columns), and last the wavefronts per SIMD asked for in the kernel without the sketch
// (beam_step_kernel_w; 0 = the compiler's own choice, which is seven at most: the step holds 106 scalar registers).
// Eight wavefronts per SIMD - every workgroup slot a compute unit has - is what the launches that wait on memory
// round trips rather than on bytes want, and the shapes that reach it without spilling a vector register ask for it
// (measured: searches of 1M x 768 1.59 -> 1.69 M queries/s, the 1M x 128 build 4.4 -> 4.1 s; at 384 columns with
// two instead of four whole rows in flight, third-loop launches 0.252 -> 0.217 ms, and the sketch kernel with one
// load in flight 0.317 -> 0.295 ms on the first loop's).  A sketch row has a quarter of the chunks, so a quarter of
// the lanes (or of the chunks per lane) covers it.  Two shapes end with the wavefronts asked for in the kernel of several
// iterations, which are one more than the compiler leaves room for (3 to 5 spilled registers): 2,400 / 10,000 queries at
// 60,000 x 1,280 1,762 -> 1,708 and 6,509 -> 6,359 us, 2,800 / 10,000 at 60,000 x 1,792 2,430 -> 2,324 and 8,228 -> 7,834.
int launch_step_by_dim(const StepArgs &s, bool aligned, int threads, size_t smem, hipStream_t st) {
    const int nchunks = s.nchunks;
    const int variant = dist_variant();
    if (nchunks > 512 || (!aligned && s.dim < 4)) launch_step<1, 64, 1, kRowScalar>(s, threads, smem, st);
    else if (!aligned) vl_launch_step_unaligned(s, threads, smem, st);
    else if (nchunks <= 16) launch_step<1, 16, 8, kRowAligned, 1, 8, 4, 5, 8, 8>(s, threads, smem, st);
    else if (nchunks <= 32 && variant == 1) launch_step<1, 32, 8, kRowAligned>(s, threads, smem, st);
    else if (nchunks <= 32) launch_step<2, 16, 4, kRowAligned, 1, 8, 4, 5, 4, 8>(s, threads, smem, st);
    else if (nchunks <= 64) launch_step<1, 64, 8, kRowAligned, 2, 8, 2, 5, 8, 8>(s, threads, smem, st);
    else if (nchunks <= 96 && variant != 1) launch_step<3, 32, 2, kRowAligned, 3, 8, 1, 8, 1, 8>(s, threads, smem, st);
    else if (nchunks <= 128) launch_step<2, 64, 8, kRowAligned, 2, 16, 2, 6, 2>(s, threads, smem, st);
    else if (nchunks <= 192) launch_step<3, 64, 2, kRowAligned, 3, 16, 1, 8, 1, 8>(s, threads, smem, st);
    else if (nchunks <= 256) launch_step<4, 64, 4, kRowAligned, 4, 16, 2, 5, 2>(s, threads, smem, st);
    else if (nchunks <= 320) launch_step<5, 64, 2, kRowAligned, 3, 32, 2, 6, 1, 0, 5>(s, threads, smem, st);
    else if (nchunks <= 384) launch_step<6, 64, 2, kRowAligned, 3, 32, 2, 6, 1>(s, threads, smem, st);
    else if (nchunks <= 448) launch_step<7, 64, 2, kRowAligned, 4, 32, 2, 5, 1, 0, 4>(s, threads, smem, st);
    else launch_step<8, 64, 2, kRowAligned, 4, 32, 2, 5, 1>(s, threads, smem, st);
    VL_LAUNCH_CHECK("beam_step_kernel");
    g_step_launches.fetch_add(1, std::memory_order_relaxed);
    return VL_OK;
}

struct BeamLayout {
    int64_t m, VL, Vt, E, head;
    int64_t off_cand_ids, off_cand_d, off_v_ids, off_v_d, off_seen, off_seen_count, off_row_quiet, off_memo_rate, off_ctrl, off_rounded, off_memo, total;
    int memo_slots;
    bool may_sketch;     // the call may bring a sketch and use it (as far as its parameters tell: not the rows' addresses)
    bool rows_meet_again;  // what meets_again says
    // the table of all distances (beam_table.hip) and the copies it is made from, over the cache
    bool use_table;
    int64_t table_columns, off_packed_queries, off_packed_vectors, off_table, table_end;
    // or the bounds of all of them (near_products.h), behind the cache
    bool use_near;
    NearPlan near_plan;
    int64_t off_near, near_end;
};

inline int64_t align256(int64_t x) { return (x + 255) & ~255ll; }

constexpr int kLeastCacheSlots = 1024;  // per row, where there is a cache

// Whether rows ask for so many candidates until their visited lists are full (asked) that they meet most vectors several
// times.  What is measured in one early iteration says little then: the share of repeats grows, and the cache stays in use.
// Measured without a share to reach, against the share:
// builds of 6,000 x 25 (asked 4.3 times the vectors) 0.84, 10,000 x 50 (2.6) 0.94, 9,000 x 128 (3.4) 0.86, 4,096 x 128 (7.5)
// 0.76, 3,000 x 64 (20) 0.92; 10,000 queries at 4,096 x 64 (3.8) 0.93, 8,000 x 128 (1.9) 1.03, 20,000 x 128 (0.8) 1.21,
// 20,000 x 50 (0.4) 1.08, 20,000 x 300 (1.7) 0.65.
// With the sketch a new candidate costs a quarter of a row, which up to 256 columns is little more than a probe.  Batches of
// 5,000 rows (degree 64, ms): 256 columns, 20,000 vectors (asked 6.1) 26.7 without a share to reach and 28.0 with the share,
// 40,000 (3.1) 30.4 and 30.1, 77,000 (1.6) 36.6 and 33.7, 150,000 (0.8) 36.5 and 31.7; 300 columns, 30,000 28.9 and 32.1, 77,000 40.6 and
// 41.8, 384 columns 29.3 and 31.6, 41.0 and 42.0, 512 columns, 77,000 44.1 and 46 to 52, 768 columns 61.7 and 65.0.
inline bool meets_again(int64_t dim, int64_t n_vectors, int64_t asked, bool sketch) {
    if (sketch && dim <= 256) return asked >= 4 * n_vectors;
    return dim <= 128 ? 2 * asked >= 5 * n_vectors : 4 * dim * asked >= 1280 * n_vectors;
}

// Whether a call is worth the distances of all its queries and vectors ahead of the loop (beam_table.hip), if it runs so many
// iterations.  Per pair and column they take some 0.02 ps as products (10,000 queries of 20,011 x 768 3.0 ms, 100,000 x 128 3.0),
// 0.05 ps as squared differences, in whole tiles of queries, and the copies that they are made from 2 ps an element; 50 us
// are for the launches and for the first iterations, which fill the queues.  An iteration then takes some 11 ps for each candidate of a row (6.8 to 15 measured), 4.5 us at
// least.  Without them it takes 7.5 us at least, and where the vectors are beyond the chip's L2s 30 ps and 0.08 for each column
// (batches of 10,000 rows of a first loop at 200,000 x 50 40, x 128 50, x 384 66, x 768 111, 100,003 x 256 55, x 1,536 210), 30
// otherwise (20,011 x 768 48); on a graph of near neighbours, where most distances are in the cache, 20 (20,011 x 768 22).
bool table_pays(const vl_beam_params *p, const BeamLayout &l, double iterations, double candidate_ps) {
    const double rows = (double)p->n_rows, candidates = rows * (double)l.m, elements = (double)p->n_vectors * (double)p->dim;
    const double in_tiles = (double)(pair_tiles(p->n_rows) * kPairTile) * elements;
    const double made = 50.0 + 0.02 * (double)p->dim + 2e-6 * elements + in_tiles * (p->metric == VL_METRIC_L2 ? 5e-8 : 2e-8);  // us
    const double with = candidates * 11e-6, without = candidates * candidate_ps * 1e-6;
    return made + iterations * (with > 4.5 ? with : 4.5) < 0.9 * iterations * (without > 7.5 ? without : 7.5);
}
// And whether it still is when the stores count: a pair is 1.1 ps to store (the partial sums that short rows leave empty included) and
// 0.0175 ps a column as products, 1.2 and 0.045 as squared differences (10,000 queries of 100,000 x 4 1.27 ms, x 32 1.65, x 128 3.2, of
// 20,011 x 256 1.14, x 768 2.9; squared differences of 100,000 x 4 1.69, x 128 6.9).  Above, which rows of some 60 columns and more
// decide, they are left out against iterations that are counted low; here these are what was measured.
//   First loops fill their visited lists (where there are no more than some thousand vectors, before).  Searches that say that they are
// long take the longer the more queries wait for each other: 10 to 60 iterations with 40, 15 to 125 with 300, 45 to 220 with 2,000 and
// more.  Searches with dense seeds, which say nothing, took 5 to 15 with queues of 10, 15 and more with longer ones (half the queue's
// length is counted on, 25 at most), and 40 ps and 0.08 a column for a candidate in the first five iterations, which fetch what they look at.
//   Without and with the distances, us.  10,000 queries with dense seeds and queues of 10, degree 64, at 4,096 x 24 569 and 270, 20,011 x 24 567
// and 542; left alone: 20,011 x 64 601 and 673, 60,000 x 24 2,567 and 2,787, 100,000 x 4 947 and 2,000; queues of 128 at 20,011 x 64 3,231
// and 2,587.  Searches that say that they are long, 10,000 queries: degree 24 at 60,000 x 16 3,014 and 2,420, degree 64 at 60,000 x 64 7,094
// and 5,498; left alone: degree 24 at 150,000 x 4 2,865 and 3,477, 400,000 x 4 2,383 and 6,697.  First loops, degree 24: 150,000 x 50 7,670
// and 4,436; left alone: 400,000 x 16 5,727 and 7,300.
struct ExpectedLoop {
    double iterations;
    double candidate_ps, first_ps;  // a candidate without the distances: in all iterations but the first five, in those
    double lookup_ps;               // with them
};
bool stores_pay(const vl_beam_params *p, const BeamLayout &l, const ExpectedLoop &e) {
    const double candidates = (double)p->n_rows * (double)l.m, elements = (double)p->n_vectors * (double)p->dim, dim = (double)p->dim;
    const double pairs = (double)(pair_tiles(p->n_rows) * kPairTile) * (double)p->n_vectors;
    const double made = 40.0 + 0.02 * dim + 2e-6 * elements + pairs * (p->metric == VL_METRIC_L2 ? 1.2e-6 + 4.5e-8 * dim : 1.1e-6 + 1.75e-8 * dim);  // us
    const double with = e.iterations * std::max(4.5, candidates * e.lookup_ps * 1e-6);
    const double without = e.iterations * std::max(7.5, candidates * e.candidate_ps * 1e-6) +
                           std::min(5.0, e.iterations) * candidates * (e.first_ps - e.candidate_ps) * 1e-6;
    return made + with < 0.95 * without;
}
ExpectedLoop expected_loop(const vl_beam_params *p, const BeamLayout &l, bool said) {
    const double most = (double)l.E / (double)l.Vt, anywhere = 30.0 + 0.08 * (double)p->dim;
    const double search = p->n_rows < 32 ? 20.0 : p->n_rows < 200 ? 30.0 : p->n_rows < 1000 ? 45.0 : 60.0;
    if (!said) return {std::min(25.0, 0.5 * (double)p->queue_length), 20.0, 40.0 + 0.08 * (double)p->dim, 11.0};
    if (p->excl_cols > 0) return {most, anywhere, anywhere, 10.0};
    return {std::min(most, search), anywhere, anywhere, 11.0};
}
//   A batch of a first loop of a build takes four fifths of the iterations that fill its visited lists and more, a search 85 to
// 95 (37 to 300 queries), few queries 30 (VL_BEAM_MANY_ITERATIONS); what a call that does not say takes is not known: 15 to 125, and
// 20 are counted on.  Batches of later loops find most distances in the cache (10,000 rows of 20,011 x 768 4.0 ms without and 5.6
// with the table, of 100,000 x 128 6.0 and 8.5).  First loops without and with the table, ms: 10,000 rows of 20,011 x 768 60.2 and 12.6, 50,000 x 768 88.2 and 17.6,
// 200,000 x 768 138.9 and 39.2, 100,003 x 1,536 263 and 40, 100,000 x 128 15.7 and 6.1, 200,000 x 50 10.8 and 6.1, 60,000 x 200 (L2)
// 72.9 and 12.5, 1,000 rows of 200,000 x 768 15.8 and 7.0, of 50,000 x 100 1.75 and 1.03.
constexpr int64_t kTableMostBytes = 16ll << 30;
bool table_use(const vl_beam_params *p, const BeamLayout &l) {
    if (p->flags & (VL_BEAM_NO_TABLE | VL_BEAM_TWO_LAUNCHES | VL_BEAM_SORT_MERGE | VL_BEAM_NO_WINDOWS | VL_BEAM_WINDOWS)) return false;
    if (l.Vt > kTableMaxVisit || l.VL <= l.Vt || l.VL > kTableMaxQueue || p->queue_length > kTableMaxQueue ||
        l.m > kTableMaxCandidates || p->excl_cols > kTableMaxExcluded || l.Vt * p->speculative_readahead > l.E || p->dim > 2048)
        return false;
    if (p->n_vectors < kPairTile || p->n_rows * pair_columns(p->n_vectors) * 4 > kTableMostBytes ||
        !vl_pair_table_fits(p->n_rows, p->n_vectors, p->dim))
        return false;
    if (p->flags & VL_BEAM_TABLE) return true;
    if ((p->flags & VL_BEAM_BOUNDS) && l.may_sketch) return false;  // (wants those)
    if ((p->flags & VL_BEAM_NO_CACHE) && !(p->flags & VL_BEAM_MANY_ITERATIONS)) return false;  // (asked for a small workspace)
    const double all = 0.8 * (double)l.E / (double)l.Vt, search = p->n_rows >= 32 ? 30 : 20;
    const double anywhere = p->n_vectors * p->dim > (8 << 20) ? 30 + 0.08 * (double)p->dim : 30;
    if (table_pays(p, l, 20, 20) && stores_pay(p, l, expected_loop(p, l, false))) return true;
    return (p->flags & VL_BEAM_MANY_ITERATIONS) && table_pays(p, l, p->excl_cols > 0 || all < search ? all : search, anywhere) &&
           stores_pay(p, l, expected_loop(p, l, true));
}

// Whether a call whose table of distances would be too large or too much work is given the products of all its queries and vectors in
// bfloat16 instead (near_products.h), where it would use the sketch: batches of a first loop, as above.  The products take 2 fs a
// column, storing them 0.4 ps a pair, the copies 1.5 ps an element; an iteration then takes 24 + 0.016 ps a column for each
// candidate, through the sketch 2 + 0.155.  Without and with, ms, 10,000 rows: 1M x 768 140 and 60, 500,000 x 1,024 200 and 61, x 1,536
// 306 and 85, x 256 55.1 and 41.4, 1M x 384 (degree 48) 43.5 and 37.9, x 256 (degree 32: left alone) 14.3 and 20.5; 1,000 rows of 1M x
// 768 15.9 and 8.8, 300 of 500,000 x 768 10.6 and 6.2.  The cache is left out: 62.8 ms for the first with it.
constexpr int64_t kNearMostBytes = 24ll << 30;
bool near_use(const vl_beam_params *p, const BeamLayout &l) {
    // (several iterations to a launch, as long as no list fills up in one)
    if (!l.may_sketch || l.use_table || p->speculative_readahead < 2 || l.Vt * p->speculative_readahead > l.E) return false;
    if (p->flags & (VL_BEAM_NO_TABLE | VL_BEAM_NO_WINDOWS | VL_BEAM_WINDOWS)) return false;  // (it runs several iterations per launch)
    if (p->n_vectors < kPairTile || l.near_plan.bytes > kNearMostBytes) return false;
    if (p->flags & VL_BEAM_BOUNDS) return true;
    const double rows = (double)p->n_rows, pairs = rows * (double)p->n_vectors, candidates = rows * (double)l.m;
    const double made = 60.0 + pairs * (2.2e-9 * (double)p->dim + 4e-7) + 1.5e-6 * (double)p->n_vectors * (double)p->dim;  // us
    const double iterations = 0.8 * (double)l.E / (double)l.Vt;
    const double saved = iterations * candidates * (0.139 * (double)p->dim - 22.0) * 1e-6;
    return (p->flags & VL_BEAM_MANY_ITERATIONS) && p->excl_cols > 0 && made <= 0.8 * saved;
}

// *circulant = 1 if the neighbours of node i + 1 are those of node i plus one, in a sample of the nodes (there are two at least).
constexpr int kCirculantNodes = 64;
__global__ __launch_bounds__(256) void circulant_graph_kernel(const int32_t *__restrict__ beams, int64_t n, int64_t width, int32_t *circulant) {
    __shared__ int other;
    if (threadIdx.x == 0) other = n < 2;
    __syncthreads();
    for (int64_t i = threadIdx.x; n >= 2 && i < kCirculantNodes * width; i += 256) {
        const int64_t node = i / width * (n - 1) / kCirculantNodes, k = i % width;
        const int32_t here = beams[node * width + k], next = beams[(node + 1) * width + k];
        if (here < 0 || here >= n || next != (here + 1 == n ? 0 : here + 1)) other = 1;
    }
    __syncthreads();
    if (threadIdx.x == 0) *circulant = !other;
}

// lean: the layout of the entry point that allocates nothing - the fused step keeps its candidates in LDS
// and runs without the distance cache, so neither gets room.
int beam_layout(const vl_beam_params *p, BeamLayout *l, bool lean = false) {
    VL_REQUIRE(p, "null params");
    VL_REQUIRE(p->n_rows >= 0 && p->dim > 0 && p->n_vectors > 0 && p->width > 0, "bad sizes");
    VL_REQUIRE(p->beam_size > 0 && p->parallel_visit_count > 0 && p->visit_queue_factor > 0 &&
                   p->exclude_factor > 0 && p->speculative_readahead > 0,
               "configuration values must be positive");
    VL_REQUIRE(p->queue_length > 0 && p->queue_length < p->queue_capacity, "queue length must be below its capacity");
    VL_REQUIRE(p->n_vectors < (1ll << 30), "ids must stay below 2^30");
    VL_REQUIRE(p->metric == VL_METRIC_COSINE || p->metric == VL_METRIC_L2, "unknown metric %lld", (long long)p->metric);
    VL_REQUIRE(p->n_rows <= kMaxBlocks, "a batch of %lld rows is too large for one call (limit %lld)",
               (long long)p->n_rows, (long long)kMaxBlocks);
    l->VL = p->visit_queue_factor * p->beam_size;                                      // ann.py:51
    l->Vt = l->VL < p->parallel_visit_count ? l->VL : p->parallel_visit_count;         // queue.py:89
    l->m = l->Vt * p->width;
    l->E = p->exclude_factor * l->VL;                                                  // ann.py:55
    l->head = p->queue_length < l->VL ? p->queue_length : l->VL;                       // queue.py:31
    l->may_sketch = (p->flags & VL_BEAM_USES_SKETCH) && !(p->flags & (VL_BEAM_TWO_LAUNCHES | VL_BEAM_SORT_MERGE)) &&
                    p->metric == VL_METRIC_COSINE && p->dim % 4 == 0 && p->dim <= 2048 && l->m <= kMaxCandidates;
    l->rows_meet_again = meets_again(p->dim, p->n_vectors, l->E * p->width, l->may_sketch);
    VL_REQUIRE(l->Vt <= kMaxVisit, "parallel_visit_count above %d is not supported", kMaxVisit);
    VL_REQUIRE(p->queue_length + l->m <= p->queue_capacity,
               "search queue capacity %lld cannot take %lld candidates after its %lld slots",
               (long long)p->queue_capacity, (long long)l->m, (long long)p->queue_length);
    VL_REQUIRE(p->queue_capacity <= kMaxRowSlots && l->VL + l->m <= kMaxRowSlots && l->E <= kMaxRowSlots,
               "queue rows above %d slots are not supported", kMaxRowSlots);
    VL_REQUIRE(p->excl_cols >= 0 && p->excl_cols <= 1024, "exclusion rows above 1024 ids are not supported here");
    int64_t o = 0;
    l->off_cand_ids = o; o = align256(o + (lean ? 0 : p->n_rows * l->m * 4));
    l->off_cand_d = o; o = align256(o + (lean ? 0 : p->n_rows * l->m * 4));
    l->off_v_ids = o; o = align256(o + p->n_rows * l->VL * 4);
    l->off_v_d = o; o = align256(o + p->n_rows * l->VL * 4);
    l->off_seen = o; o = align256(o + p->n_rows * l->E * 4);
    l->off_seen_count = o; o = align256(o + p->n_rows * 4);
    l->off_row_quiet = o; o = align256(o + p->n_rows * 4);
    l->off_memo_rate = o; o = align256(o + p->n_rows * 4);
    l->off_ctrl = o; o = align256(o + (int64_t)sizeof(BeamCtrl));
    // the query rows rounded for the sketch, for calls that say they bring one
    l->off_rounded = o; o = align256(o + ((p->flags & VL_BEAM_USES_SKETCH) && !lean ? p->n_rows * sketch_query_bytes(p->dim) : 0));
    // per-row cache of evaluated (id, distance) pairs: 128 slots per candidate of one iteration,
    // 1Ki..64Ki per row, the whole table at most 8 GiB (measured at 1M x 768: 16Ki -> 64Ki slots cuts the
    // rows fetched in the second optimisation loop by 30 %, 256Ki adds little)
    static const int memo_env = [] {
        const char *e = getenv("VL_BEAM_MEMO");
        return e ? atoi(e) : -1;
    }();
    // ... and no more than 512 per slot of the search queue: a search with a short queue ends after few
    // iterations, fills little of a large table and would pay for clearing it on every call
    int64_t want = 128 * l->m < 512 * p->queue_length ? 128 * l->m : 512 * p->queue_length;
    int slots = vl_next_pow2(want > 65536 ? 65536 : want);
    // ... and no more than the vectors need (a quarter of them over, for the sake of collisions): a build of 6,007 x 384
    // 15.3 ms with 64Ki slots, 13.9 with 8Ki, 19.1 with 4Ki; of 4,096 x 128 5.10 with 32Ki, 4.86 with 8Ki, 5.12 with 4Ki; of
    // 20,011 x 768 130.1 with 64Ki, 128.2 with 32Ki, 160.8 with 16Ki
    const int64_t most = p->n_vectors + p->n_vectors / 4;
    if (slots > most) slots = vl_next_pow2(most);
    // ... and of rows of up to 512 bytes that meet few vectors again 16 per candidate: such a row is fetched again for little
    // more than a probe, and clearing and spreading the table costs more.  Us with 128 slots per candidate (a whole table) and
    // with 16: 10,000 queries at 1M x 128 1,991 and 1,711, at 100,000 x 128 5,389 and 5,151, at 60,000 x 50 5,969 and 5,693,
    // builds of 100,000 x 128 275 and 269 ms, a batch of a first loop at 300,000 x 96 15.2 and 14.9.  Not with longer rows: a batch of
    // 100,000 x 200 (no clusters, m = 512) 124.4 ms with 64Ki, 127.3 with 32Ki, 131.6 with 8Ki.
    if (p->dim <= 128 && !l->rows_meet_again) {
        const int enough = vl_next_pow2(16 * l->m);
        if (slots > enough) slots = enough;
    }
    if (slots < kLeastCacheSlots) slots = kLeastCacheSlots;
    if (slots > 65536) slots = 65536;
    while (slots > kLeastCacheSlots && p->n_rows * (int64_t)slots * 8 > (8ll << 30)) slots >>= 1;
    if (memo_env >= 0) slots = memo_env;
    if (lean || (p->flags & VL_BEAM_NO_CACHE)) slots = 0;
    l->memo_slots = slots;
    l->off_memo = o; o = align256(o + p->n_rows * (int64_t)slots * 8);
    l->total = o;
    l->use_table = !lean && table_use(p, *l);
    l->table_columns = l->off_packed_queries = l->off_packed_vectors = l->off_table = l->table_end = 0;
    if (l->use_table) {
        l->table_columns = pair_columns(p->n_vectors);
        l->off_packed_queries = l->off_memo;
        l->off_packed_vectors = l->off_packed_queries + pair_packed_bytes(p->n_rows, p->dim);
        l->off_table = l->off_packed_vectors + pair_packed_bytes(l->table_columns, p->dim);
        l->table_end = l->off_table + p->n_rows * l->table_columns * 4;
    }
    l->use_near = false;
    l->off_near = l->near_end = 0;
    if (!lean && l->may_sketch) {
        l->near_plan = vl_near_plan(p->n_rows, p->n_vectors, p->dim);
        l->use_near = near_use(p, *l);
        if (l->use_near) {
            l->off_near = l->total;
            l->near_end = l->off_near + l->near_plan.bytes;
        }
    }
    return VL_OK;
}

}  // namespace

VL_EXPORT int64_t vl_beam_workspace_bytes(const vl_beam_params *p) {
    BeamLayout l;
    int rc = beam_layout(p, &l);
    return rc < 0 ? rc : std::max(l.total, std::max(l.table_end, l.near_end));
}

namespace {
bool profiling() {
    std::lock_guard<std::mutex> hold(g_prof_mutex);
    return g_prof.enabled != 0;
}
}  // namespace

VL_EXPORT int vl_beam_ahead(const vl_beam_params *p) {
    BeamLayout l;
    int rc = beam_layout(p, &l);
    if (rc < 0) return rc;
    const bool said = (p->flags & VL_BEAM_MANY_ITERATIONS) != 0, prof = profiling();
    if (l.use_table) return prof && !said && !(p->flags & VL_BEAM_TABLE) ? 0 : VL_BEAM_TABLE;
    if (l.use_near) return VL_BEAM_BOUNDS;
    // (a look at the graph waits for the stream: not for a few rows)
    if (prof || said || (p->flags & (VL_BEAM_NO_CACHE | VL_BEAM_KNOWN_GRAPH)) || p->excl_cols == 0 || p->n_rows < kComputeUnits) return 0;
    vl_beam_params of_first_loop = *p;
    of_first_loop.flags |= VL_BEAM_MANY_ITERATIONS;
    rc = beam_layout(&of_first_loop, &l);
    return rc < 0 ? rc : l.use_table || l.use_near ? VL_BEAM_MANY_ITERATIONS : 0;
}

VL_EXPORT int vl_circulant_graph(const int32_t *beams, int64_t n_vectors, int64_t width, int32_t *circulant, void *stream) {
    VL_REQUIRE(n_vectors > 0 && width > 0, "bad sizes");
    VL_REQUIRE(beams && circulant, "null pointer");
    hipLaunchKernelGGL(circulant_graph_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream, beams, n_vectors, width, circulant);
    VL_LAUNCH_CHECK("circulant_graph_kernel");
    return VL_OK;
}

namespace {

__global__ void beam_empty_status_kernel(int32_t *status) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        status[0] = 1;
        status[1] = 0;
    }
}

__global__ void beam_status_kernel(const BeamCtrl *c, int iterations, int R, int32_t *status) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    int ended = c->stop, t = c->ended_after;
    if (!ended && iterations % R == 0 && c->changed[(iterations / R) & 63] == 0) {
        ended = 1;  // the last launch was a checking iteration that found every row quiet
        t = iterations;
    }
    status[0] = c->error ? -1 : ended;  // -1: a row's state was impossible (the scratch memory was shared with another call)
    status[1] = ended ? t : iterations;
}

// After a refused table: the launch that was enqueued behind the refused one may be an ordinary one, which takes the check that
// nothing ran up to for one that found the batch quiet and ends the loop.  The loop begins again.
__global__ void beam_resume_kernel(BeamCtrl *c) {
    if (threadIdx.x == 0 && blockIdx.x == 0) c->stop = c->ended_after = c->refused_at = 0;
}

// The loop itself.  fixed_iterations == 0: run until a progress check finds the batch quiet, reading the
// flag on the host every speculative_readahead iterations; returns the iteration count.  fixed_iterations
// > 0: enqueue exactly that many iterations and return 0 without ever waiting for the device - once a
// check finds the batch quiet the remaining launches do nothing (beam_gate) - then one small kernel writes
// status_out[0] = 1 if the loop ended within them (else 0) and status_out[1] = the iteration count.
int64_t beam_loop(const vl_beam_params *p, BeamLayout l, const float *queries, const float *vectors,
                  const int32_t *beams, int32_t *q_ids, float *q_dists, const int32_t *exclude, void *workspace,
                  int64_t workspace_bytes, int64_t fixed_iterations, int32_t *status_out, void *stream,
                  const uint8_t *sketch = nullptr) {
    int rc;
    VL_REQUIRE(queries && vectors && beams && q_ids && q_dists && workspace, "null pointer");
    VL_REQUIRE(((uintptr_t)workspace & 255) == 0, "workspace must be 256-byte aligned");
    // A workspace sized for the same rows of a table with more or fewer vectors or columns serves: the cache, which lies at
    // the end, takes the slots that fit.  Refused is what is too small for a table of any size.
    while (l.total > workspace_bytes && l.memo_slots > kLeastCacheSlots) {
        l.memo_slots >>= 1;
        l.total = align256(l.off_memo + p->n_rows * (int64_t)l.memo_slots * 8);
    }
    if (workspace_bytes < l.total) {
        vl_set_error("workspace of %lld bytes is smaller than the %lld needed", (long long)workspace_bytes,
                     (long long)l.total);
        return VL_ERR_WORKSPACE;
    }
    VL_REQUIRE(p->n_rows * (l.VL > l.m ? l.VL : l.m) < (1ll << 40), "batch too large");
    VL_REQUIRE(p->n_rows * (int64_t)l.VL < (1ll << 31), "batch too large: %lld rows with visit queues of %d slots",
               (long long)p->n_rows, (int)l.VL);
    hipStream_t st = (hipStream_t)stream;
    if (fixed_iterations == 0) {  // refused before anything is recorded: the loop waits for what its launches find
        hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(st, &capturing) != hipSuccess) (void)hipGetLastError();
        if (capturing != hipStreamCaptureStatusNone) {
            vl_set_error("this call waits for its stream and cannot be captured into a graph "
                         "(vl_closest_vectors_noalloc can)");
            return VL_ERR_HIP;
        }
    }
    char *ws = (char *)workspace;
    int32_t *cand_ids = (int32_t *)(ws + l.off_cand_ids);
    float *cand_d = (float *)(ws + l.off_cand_d);
    int32_t *v_ids = (int32_t *)(ws + l.off_v_ids);
    float *v_d = (float *)(ws + l.off_v_d);
    int32_t *seen = (int32_t *)(ws + l.off_seen);
    int32_t *seen_count = (int32_t *)(ws + l.off_seen_count);
    int32_t *row_quiet = (int32_t *)(ws + l.off_row_quiet);
    BeamCtrl *ctrl = (BeamCtrl *)(ws + l.off_ctrl);

    uint64_t *memo = (uint64_t *)(ws + l.off_memo);
    MergeArgs a;
    a.ctrl = ctrl; a.readahead = (int)p->speculative_readahead; a.n_rows = p->n_rows;
    a.cand_ids = cand_ids; a.cand_d = cand_d; a.m = (int)l.m;
    a.q_ids = q_ids; a.q_d = q_dists; a.cap = (int)p->queue_capacity; a.L = (int)p->queue_length;
    a.Ps = vl_next_pow2(a.cap);
    a.excl = p->excl_cols > 0 ? exclude : nullptr; a.excl_cols = a.excl ? (int)p->excl_cols : 0;
    a.v_ids = v_ids; a.v_d = v_d; a.VL = (int)l.VL; a.Vt = (int)l.Vt; a.Pv = vl_next_pow2(l.VL + l.m);
    a.seen = seen; a.seen_count = seen_count; a.E = (int)l.E;
    const bool per_query = (p->flags & VL_BEAM_PER_QUERY_STOP) != 0;
    a.row_quiet = per_query ? row_quiet : nullptr;
    a.Pc = vl_next_pow2(l.m);
    if (a.Pc < 2) a.Pc = 2;
    // VL_BEAM_MERGE=sort selects the full-row-sort form of the merge step (exact for queue rows in any state)
    static const bool sort_merge_env = [] {
        const char *e = getenv("VL_BEAM_MERGE");
        return e && e[0] == 's';
    }();
    const bool use_sort_merge = sort_merge_env || (p->flags & VL_BEAM_SORT_MERGE);
    const bool aligned = (p->dim % 4 == 0) && (((uintptr_t)queries | (uintptr_t)vectors) % 16 == 0);
    // VL_BEAM_WINDOWS / VL_BEAM_NO_WINDOWS in flags, or VL_BEAM_WINDOW=1 / 0 in the environment: windows always / never.
    static const int window_env = [] {
        const char *e = getenv("VL_BEAM_WINDOW");
        return e ? atoi(e) : -1;
    }();
    const bool all_windows = window_env >= 0 ? window_env != 0 : (p->flags & VL_BEAM_WINDOWS) != 0;
    const bool no_windows = window_env >= 0 ? window_env == 0 : (p->flags & VL_BEAM_NO_WINDOWS) != 0;
    // Threads per row.  A few rows want the wavefronts: idle ones share in the fetch.  Rows that fill the chip want as many of
    // them in flight as it holds: 128 threads, unless a row has more than 320 candidates in an iteration (ms of a build of
    // 8,000 x 200 with m = 256 / 288 / 384 / 512, 128 and 256 threads: 17.7 and 19.2, 18.8 and 20.3, 27.3 and 23.9, 29.6 and
    // 22.2, with the sketch (8,000 x 384) 20.7 and 23.2, 20.3 and 22.9, 39.0 and 37.3, 48.5 and 39.3).
    // Few are the rows that a compute unit holds at once with 256 threads: six, and four of the shapes whose registers leave four
    // wavefronts per SIMD (aligned rows of 385 to 512 columns without the sketch, rows of more than 768).  Time with 128
    // threads over time with 256 at 4 / 5 / 6 / 7 rows per compute unit: queries at 20,011 x 50 (m = 96) 1.08 / 1.05 / 1.04 /
    // 0.73, 8,000 x 130 (96) 1.29 / 1.27 / 1.25 / 0.84, 50,000 x 384 (192) 1.05 / 1.04 / 1.02 / 0.82, 100,000 x 768 (256) 1.10 / 1.09 /
    // 1.06 / 0.94, 60,000 x 200 (256) 1.12 / 1.08 / 1.08 / 0.89, 100,000 x 512 (256) 1.13 / 0.87 / 0.84 / 0.84, 100,000 x 1,536 (256)
    // 1.06 / 0.88 / 0.88 / 0.86, rows of a first loop at 60,000 x 50 (288) 1.39 / 1.35 / 1.32 / 0.85, at 60,000 x 768 with the sketch
    // (256) 1.21 / 1.11 / 1.04 / 0.87.
    // Aligned rows with up to 128 candidates, which dense seeds start near their neighbours, fetch less, and fewer of them are few: at
    // 1 / 2 / 3 / 4 per compute unit 4,096 x 128 1.04 / 1.04 / 1.02 / 1.00, 100,000 x 128 in clusters of 977 1.00 / 0.99 / 0.98 / 0.96,
    // 11,717 x 96 0.98 / 0.98 / 0.98 / 0.94; at 4 / 5 / 6 60,000 x 200 in clusters of 244 0.96 / 0.94 / 0.93, x 384 0.96 / 0.95 / 0.94, x
    // 768 0.97 / 0.96 / 0.96.  (Without clusters more would do: 20,000 x 200 1.20 / 1.17 / 1.14, x 384 1.08 / 1.00 / 0.95, x 768 1.01 / 0.97 / 0.97.)
    // With the sketch and more than 768 columns (one iteration per launch) 256 threads are the sooner at 5 / 7 / 9 / 12 / 39 rows per
    // compute unit too: a first loop's rows at 60,000 x 1,024 (m = 256) 1.02 / 1.03 / 1.06 / 1.08 / 1.06, (m = 288) 1.01 at 5,
    // 1.05 at 9, 1.06 at 39, at 60,000 x 1,536 (256) 1.05 at 9, 1.06 at 39.
    const int64_t rows_per_cu = (p->n_rows + kComputeUnits - 1) / kComputeUnits;
    const bool holds_six = p->dim <= 768 && !(aligned && !sketch && p->dim > 384 && p->dim <= 512);
    const int64_t few = l.m <= 128 && aligned ? 2 : holds_six ? 6 : 4;
    static const int merge_threads_env = [] {
        const char *e = getenv("VL_BEAM_MERGE_THREADS");
        return e ? atoi(e) : 0;
    }();
    const int merge_threads = merge_threads_env ? merge_threads_env
                              : ((l.m > 320 || rows_per_cu <= few || (sketch && p->dim > 768)) ? 256 : 128);
    const int Pmax = a.Ps > a.Pv ? a.Ps : a.Pv;
    const size_t smem = use_sort_merge
        ? (size_t)Pmax * 8 + (size_t)a.L * 4 + (size_t)a.E * 8 + (size_t)a.excl_cols * 4
        : (size_t)a.Pc * 16 + (size_t)(a.L + a.VL) * 8 + (size_t)a.E * 8 + (size_t)a.excl_cols * 4 + (size_t)a.m + 16;
    // the LDS of a row that has visited all it can
    const size_t smem_step = row_layout(a.m, a.L, a.VL, row_hash_slots(a.E, a.m, false), a.excl_cols, false).bytes;
    const size_t smem_window = row_layout(a.m, a.L, a.VL, row_hash_slots(a.E, a.m, true), a.excl_cols, true).bytes;
    // VL_BEAM_FUSED=0 runs an iteration as two launches (expand, merge) instead of the fused step
    static const bool fused_env = [] {
        const char *e = getenv("VL_BEAM_FUSED");
        return !(e && e[0] == '0');
    }();
    const bool use_fused = fused_env && !use_sort_merge && merge_threads != 64 && !(p->flags & VL_BEAM_TWO_LAUNCHES);
    VL_REQUIRE((use_fused ? smem_step : smem) + 2048 <= kLdsPerCu, "queues of this size need %zu bytes of LDS (a compute unit has %zu)",
               use_fused ? smem_step : smem,
               kLdsPerCu);
    VL_REQUIRE(!per_query || use_fused, "the per-query stop is only built into the fused step");
    if (!use_fused) {
        if (use_sort_merge) VL_HIP(vl_allow_lds(beam_merge_kernel, smem));
        else if (merge_threads == 64) VL_HIP(vl_allow_lds(beam_merge2_kernel<64>, smem));
        else if (merge_threads == 128) VL_HIP(vl_allow_lds(beam_merge2_kernel<128>, smem));
        else VL_HIP(vl_allow_lds(beam_merge2_kernel<256>, smem));
    }
    StepArgs step;
    step.queries = queries; step.vectors = vectors; step.beams = beams; step.n_vectors = p->n_vectors;
    step.dim = (int)p->dim; step.nchunks = (int)((p->dim + 3) / 4); step.width = (int)p->width;
    step.width_magic = (uint32_t)((1ull << 32) / (uint64_t)p->width + 1);  // not used for width 1 (it does not fit)
    step.l2 = p->metric == VL_METRIC_L2;
    step.memo = l.memo_slots > 0 ? memo : nullptr;
    step.memo_rate = (int32_t *)(ws + l.off_memo_rate);  // written in iteration kMemoDecide, read after it
    {
        // break-even share of hits, measured on 512-byte rows at about 0.4 and scaled with the row size
        static const int rate_env = [] {
            const char *e = getenv("VL_BEAM_MEMO_MIN_RATE");
            return e ? atoi(e) : -1;
        }();
        const int64_t row_bytes = 4 * p->dim;
        int64_t r = (205ll * 256) / row_bytes;
        if (l.rows_meet_again) r = 0;
        step.memo_min_rate = rate_env >= 0 ? rate_env : (int)(r > 255 ? 255 : r);
    }
    // The sketch serves the cosine distance of 16-byte aligned rows in the fused step; other calls ignore it.
    step.sketch = (sketch && !step.l2 && aligned && use_fused && p->dim <= 2048 && l.m <= kMaxCandidates) ? sketch : nullptr;
    VL_REQUIRE(!step.sketch || (p->flags & VL_BEAM_USES_SKETCH),
               "a call with a sketch needs VL_BEAM_USES_SKETCH in flags (and a workspace sized with it)");
    step.rounded_queries = (const uint8_t *)(ws + l.off_rounded);
    step.rounded_query_bytes = sketch_query_bytes(p->dim);
    step.near_values = nullptr;
    step.sketch_tails = sketch ? sketch + sketch_tails_offset(p->n_vectors, p->dim) : nullptr;
    step.sketch_chunks = (int)sketch_data_chunks(p->dim);
    step.window = 0;
    step.hash_slots = 0;  // set for each launch (size_set)
    step.report = nullptr;
    step.memo_shift = 32;
    if (step.memo) {
        int lg = 0;
        while ((1 << lg) < l.memo_slots) ++lg;
        VL_REQUIRE((1 << lg) == l.memo_slots && lg >= 4, "memo slots must be a power of two, 16 or more");
        step.memo_shift = 32 - lg;
    }
    // with a sketch every row starts out using it (and the cache, when there is one)
    const bool sketch_from_start = step.sketch != nullptr;
    // (neither with the table of all distances)
    const bool prof = fixed_iterations == 0 && profiling();
    bool table = use_fused && !no_windows && l.use_table && l.table_end <= workspace_bytes;
    // what is counted are the rows that are fetched: a profiled call has the table only where it is asked for
    if (prof && !(p->flags & (VL_BEAM_MANY_ITERATIONS | VL_BEAM_TABLE))) table = false;
    const bool near = step.sketch && !no_windows && l.use_near && l.near_end <= workspace_bytes;
    const int64_t all_slots = p->n_rows * (int64_t)l.memo_slots;
    const bool cleared = !table && !near;  // the cache, with the loop's state
    auto clear_cache = [&]() -> int {
        if (all_slots > 0) {
            hipLaunchKernelGGL(beam_memo_clear_kernel, dim3(4096), dim3(256), 0, st, memo, all_slots);
            VL_LAUNCH_CHECK("beam_memo_clear_kernel");
        }
        return VL_OK;
    };
    auto make_ready = [&](bool clear) -> int {  // what a loop without the table needs
        if (sketch_from_start) {
            rc = vl_launch_sketch_queries(queries, p->n_rows, p->dim, (uint8_t *)(ws + l.off_rounded), st);
            if (rc < 0) return rc;
        }
        return clear ? clear_cache() : VL_OK;
    };
    {
        int64_t n = p->n_rows * l.VL;
        if (n < kBeamStripes) n = kBeamStripes;
        if (n < p->n_rows) n = p->n_rows;
        int64_t blocks = (n + kQueueThreads - 1) / kQueueThreads;
        const bool clear = cleared && all_slots > 0;
        if (clear) {  // eight slots a thread, up to 4,096 workgroups
            const int64_t wanted = (all_slots + 8 * kQueueThreads - 1) / (8 * kQueueThreads);
            blocks = std::max(blocks, std::min<int64_t>(wanted, 4096));
        }
        hipLaunchKernelGGL(beam_init_kernel, dim3((unsigned)blocks),
                           dim3(kQueueThreads), 0, st, ctrl, p->n_rows, q_ids, q_dists, (int)p->queue_capacity,
                           (int)l.head, v_ids, v_d, (int)l.VL, seen_count, row_quiet, (int32_t *)(ws + l.off_memo_rate),
                           sketch_from_start ? (256 | (1 << 16)) : 256, sketch_from_start ? (int)p->n_rows : 0,
                           clear ? memo : nullptr, all_slots);
        VL_LAUNCH_CHECK("beam_init_kernel");
    }
    if (!table) {
        rc = make_ready(!cleared && !near);
        if (rc < 0) return rc;
        if (near) step.memo = nullptr;
    }

    const int R = (int)p->speculative_readahead;
    // Several iterations per launch (beam_row): the R iterations between two progress checks run in one launch while no
    // visited list can fill up in them, i.e. while Vt * (last iteration) <= E; the stretch after that runs one iteration
    // per launch.  Measured against one iteration per launch: searches of 256 queries at 4,096 x 128 1,500 -> 1,004 us,
    // 1,000 at 100,003 x 1,536 1,803 -> 1,253, 10,000 at 1M x 128 2,690 -> 2,057, 10,000 at 1M x 768 3,790 -> 3,310 to 3,640 us;
    // builds of 4,096 x 128 8.5 -> 6.9 ms, 100,000 x 128 320 -> 296 ms.
    // With the sketch a window fits a compute unit six times, the one-iteration kernel eight times.  Rows that come from
    // HBM do not need those (a batch of the first loop at 1M x 768: 148 -> 140 ms, 1M x 384 49.4 -> 47.2, 50,000 x 768
    // 93.7 -> 91.2); while the table fits the chip's L2s (8 x 4 MiB) the launches wait on round trips and do (builds of
    // 20,011 x 768: 133 ms without, 143 with windows, 30,000 x 768 254 and 262).  From 769 columns on the sketch window
    // spills vector registers, and what it saves in launches goes there: a batch of the first loop at 600,000 x 2,048 534.8
    // ms without and 541.9 with windows, 100,000 x 2,048 356 and 362, 600,000 x 1,536 373.1 and 373.5, 600,000 x 1,024 228.9
    // and 228.8, builds of 24,000 x 1,536 199.9 and 205.0, 50,000 x 1,024 510 and 514 (600,000 x 512: 121.0 and 114.9).
    // Without a sketch windows are faster for every length of a row (10,000 queries at 150,000 rows of 512 columns 7.34 ->
    // 6.68 ms, 1,024 9.26 -> 7.79, 1,536 9.91 -> 9.15, 2,048 12.17 -> 11.74; 1,000 queries 1.46 -> 0.95, 1.67 -> 1.12,
    // 1.82 -> 1.27, 2.00 -> 1.83).
    constexpr int64_t kL2Bytes = 32 << 20;
    const bool sketch_window = all_windows || (p->dim <= 768 && p->n_vectors * sketch_row_bytes(p->dim) > kL2Bytes);
    const bool use_window = use_fused && !no_windows && R >= 2 && row_hash_slots_most(a.E, a.m) < 0xffff &&
                            smem_window + 2048 <= kLdsPerCu;
    // Threads of a launch.  With 128 a compute unit holds twelve rows (sixteen of one iteration), where their LDS leaves room
    // for so many, and that shrinks as the visited lists grow: at queue 128, m = 256 and E = 960 eleven rows fit at first and
    // eight in the end, sixteen wavefronts, where six rows of 256 threads are 24.  So a call whose rows do not all fit goes
    // on with 256 threads once no more than three quarters do, or once they do not if both take two rounds (and a compute
    // unit holds six of 256).  Early launches, and with them searches that end early, keep the rows.
    // 128 threads throughout / 256 / this (ms), degree 64: 2,800 queries at 20,000 x 256 14.0 / 11.3 / 11.3, x 768 29.0 / 26.1 /
    // 26.3; 4,096 at x 128 10.7 / 9.7 / 10.0, x 384 21.5 / 20.7 / 20.8, x 512 29.3 / 26.5 / 27.9, x 902 44.0 / 45.8 / 44.9, x 1,282
    // 67.8 / 59.6 / 64.6; 10,000 at x 64 15.9 / 15.4 / 15.4, x 130 38.5 / 34.5 / 35.5; at 60,000 x 128 in clusters of 244, which end early,
    // 3.46 / 4.08 / 3.46, x 768 5.47 / 6.02 / 5.48, in clusters of 977 19.48 / 19.88 / 19.48.  (At five sixths, ten rows, the
    // clusters pay for it: 3.80, 5.83, 19.91.)  Not with the sketch, where it made no difference (2,800 rows of a first loop at
    // 60,000 x 768 12.97 and 13.02).
    auto threads_of = [&](int64_t last_iteration, bool windowed) -> int {
        if (merge_threads != 128) return 256;
        if (merge_threads_env || step.sketch) return 128;
        const int64_t visited = l.Vt * last_iteration < l.E ? l.Vt * last_iteration : l.E;
        const size_t bytes = row_layout(a.m, a.L, a.VL, row_hash_slots(visited, a.m, windowed), a.excl_cols, windowed).bytes + 128;
        const int64_t fit = (int64_t)(kLdsPerCu / ((bytes + kLdsGranule - 1) / kLdsGranule * kLdsGranule)), most = windowed ? 12 : 16;
        return rows_per_cu > fit && (4 * fit <= 3 * most || (holds_six && rows_per_cu <= 12)) ? 256 : 128;
    };
    // A launch's LDS.  The visited ids of its last iteration and the candidates share the hash set, and the emptier it is
    // the sooner each finds its place, so it takes what LDS the workgroups that a compute unit can hold (or that there are)
    // leave it.  Where a batch is one round of such workgroups, their share is counted in the pieces that LDS is handed out in:
    // else ten, eleven or twelve that were to share a compute unit take a piece more each than there is, and the last rows
    // run in a round of their own.  2,400 rows (ten per compute unit), share in bytes and in pieces: queries at 100,000 x 384
    // 2,282 and 1,946 us, at 60,000 x 200 1,632 and 1,462, batches of a first loop at 60,000 x 768 (degree 32) 13.4 and 11.4 ms,
    // at 60,000 x 130 14.2 and 9.0; 2,800 (eleven) at 60,000 x 384 (degree 24) 8.0 and 7.3 ms, 60,000 x 256 searched 3,112 and
    // 3,155 us.  A batch of more rounds does better with the larger set (10,000 rows at 60,000 x 768 44.5 and 45.0 ms).
    auto size_set = [&](int64_t last_iteration, bool windowed, int threads) -> size_t {
        const int64_t visited = l.Vt * last_iteration < l.E ? l.Vt * last_iteration : l.E;
        const int waves = threads / kWave;
        const int64_t most_resident = (windowed ? 4 * 6 : 4 * 8) / waves;
        const int64_t share = rows_per_cu <= most_resident ? (int64_t)(kLdsPerCu / kLdsGranule / rows_per_cu * kLdsGranule)
                                                          : (int64_t)kLdsPerCu / most_resident;
        const int least = row_hash_slots(visited, a.m, windowed), most = row_hash_slots_most(visited, a.m);
        const int64_t room = share - 1024 - row_layout(a.m, a.L, a.VL, 0, a.excl_cols, windowed).bytes;
        int64_t slots = (room < 0 ? 0 : room) / 4;
        slots = slots > most ? most : slots;
        step.hash_slots = (int)(slots < least ? least : slots) & ~3;
        return row_layout(a.m, a.L, a.VL, step.hash_slots, a.excl_cols, windowed).bytes;
    };
    auto window_fits = [&](int64_t first_iteration) { return use_window && l.Vt * (first_iteration + R - 1) <= l.E; };
    if (fixed_iterations > 0) {
        VL_REQUIRE(use_fused, "a fixed number of iterations is only built for the fused step");
        step.count_evals = 0;
        for (int64_t t = 1; t <= fixed_iterations;) {
            a.iter = (int)t;
            step.m = a;
            const bool windowed = window_fits(t) && (t - 1) % R == 0 && t + R - 1 <= fixed_iterations;
            step.window = windowed ? R : 0;
            const int64_t last = windowed ? t + R - 1 : t;
            const int threads = threads_of(last, windowed);
            rc = launch_step_by_dim(step, aligned, threads, size_set(last, windowed, threads), st);
            if (rc < 0) return rc;
            t += windowed ? R : 1;
        }
        hipLaunchKernelGGL(beam_status_kernel, dim3(1), dim3(64), 0, st, ctrl, (int)fixed_iterations, R, status_out);
        VL_LAUNCH_CHECK("beam_status_kernel");
        return 0;
    }
    step.count_evals = prof ? 1 : 0;
    EventSet events;
    hipEvent_t *ev = events.ev;
    BeamProfile mine;
    if (prof) {
        VL_REQUIRE(R <= 64, "profiling supports speculative_readahead up to 64");
        rc = events.create(3 * R);
        if (rc < 0) return rc;
    }
    // A row expands real nodes in an unbroken run of iterations from the first one, each of
    // which adds at least one id to its visited list of E slots; once no row expands, no
    // queue changes and the next check ends the loop.  More iterations than that mean the
    // control block was overwritten while the loop ran (a workspace shared by two calls).
    const int64_t t_limit = l.E + l.VL + 2 * (int64_t)R + 2;
    // One launch serves the whole batch: the kernel that can read the sketch is launched while most rows of the
    // batch still use it.  A row gives the sketch up when it does not pay (counted on the device, read by the
    // host at its regular progress check); in the other kernel such a row goes on as it would without a sketch.
    const uint8_t *sketch_table = step.sketch;
    int sketch_rows = sketch_from_start ? (int)p->n_rows : 0;
    int64_t t = 0;
    // A call that is not profiled keeps the GPU busy across its progress checks: the launch after a checking iteration
    // is enqueued before the host knows what the check found - it does nothing if the check ended the loop (beam_gate)
    // - and reports it from its first workgroup.
    ReportSlot<StreamOfCall> slot(StreamOfCall{st});
    const bool ahead = use_fused && !prof && slot.get() != nullptr;
    step.report = ahead ? slot.get() : nullptr;
    TableStepArgs by_table;
    by_table.beams = beams; by_table.n_vectors = p->n_vectors; by_table.width = step.width; by_table.width_magic = step.width_magic;
    by_table.table = (uint32_t *)(ws + l.off_table); by_table.columns = l.table_columns; by_table.unordered = &ctrl->unordered;
    by_table.enter = 1; by_table.window = R; by_table.count_wanted = step.count_evals; by_table.report = step.report;
    bool near_made = false;
    auto launch_next = [&]() -> int {  // the fused launch that follows iteration t; moves t on
        if (table && t % R == 0 && l.Vt * (t + R) <= l.E) {
            if (by_table.enter) {
                rc = vl_launch_pair_table(queries, p->n_rows, vectors, p->n_vectors, p->dim, (int)p->metric,
                                          (uint8_t *)(ws + l.off_packed_queries), (uint8_t *)(ws + l.off_packed_vectors),
                                          by_table.table, by_table.columns, &ctrl->unordered, st);
                if (rc < 0) return rc;
                step.memo = nullptr;  // the table lies over the cache
            }
            a.iter = (int)(t + 1);
            by_table.m = a;
            t += R;
            by_table.raise_fill = l.Vt * (t + R) > l.E;
            rc = vl_launch_table_step(by_table, st);
            by_table.enter = 0;
            g_step_launches.fetch_add(1, std::memory_order_relaxed);
            return rc;
        }
        // (the iterations behind those of the table do without both)
        const bool want_sketch = sketch_table && !table && 2 * (int64_t)sketch_rows >= p->n_rows;
        const bool by_products = near && want_sketch && t % R == 0 && window_fits(t + 1);
        const bool windowed = by_products || (window_fits(t + 1) && t % R == 0 && (!want_sketch || sketch_window));
        step.near_values = nullptr;
        // (the cache is worth less than its probes with them, and is there again for rows that gave the bounds up)
        if (near && !by_products && !step.memo && l.memo_slots > 0 && !(near_made && want_sketch)) {
            rc = clear_cache();
            if (rc < 0) return rc;
            step.memo = memo;
        }
        if (by_products) {
            uint8_t *const at = (uint8_t *)ws + l.off_near;
            if (!near_made) {
                rc = vl_launch_near_products(l.near_plan, queries, p->n_rows, vectors, p->n_vectors, p->dim, at, st);
                if (rc < 0) return rc;
                near_made = true;
            }
            step.near_values = (const uint16_t *)(at + l.near_plan.off_values);
            step.near_columns = (const uint32_t *)(at + l.near_plan.off_columns);
            step.near_queries = (const NearQuery *)(at + l.near_plan.off_queries);
            step.near_pitch = l.near_plan.columns;
        }
        a.iter = (int)(t + 1);
        step.m = a;
        // (the sketch kernel also for a first window: its rows leave the sketch alone in iteration 1)
        step.sketch = ((windowed || t > 0) && want_sketch) ? sketch_table : nullptr;
        step.window = windowed ? R : 0;
        t += windowed ? R : 1;
        const int threads = threads_of(t, windowed);
        return launch_step_by_dim(step, aligned, threads, size_set(t, windowed, threads), st);
    };
    int64_t checked = 0;  // iterations up to the last progress check
    for (;;) {
        int launches = 0;  // of this stretch between two progress checks
        slot.launching();
        checked += R;
        while (t < checked) {
            const int at = launches++;
            if (prof) VL_HIP(hipEventRecord(ev[3 * at], st));
            if (use_fused) {
                rc = launch_next();
                if (rc < 0) return rc;
                if (prof) VL_HIP(hipEventRecord(ev[3 * at + 1], st));
                continue;
            }
            a.iter = (int)++t;
            rc = vl_launch_expand(queries, p->n_rows, vectors, p->n_vectors, p->dim, nullptr, v_ids, l.Vt, beams,
                                  p->n_vectors, p->width, l.m, cand_ids, cand_d, ctrl, (int)t, R, (int)l.E, l.VL,
                                  prof ? 1 : 0, memo, l.memo_slots, (int)p->metric, st);
            if (rc < 0) return rc;
            if (prof) VL_HIP(hipEventRecord(ev[3 * at + 1], st));
            if (use_sort_merge)
                hipLaunchKernelGGL(beam_merge_kernel, dim3((unsigned)p->n_rows), dim3(kQueueThreads), smem, st, a);
            else if (merge_threads == 64)
                hipLaunchKernelGGL(beam_merge2_kernel<64>, dim3((unsigned)p->n_rows), dim3(64), smem, st, a);
            else if (merge_threads == 128)
                hipLaunchKernelGGL(beam_merge2_kernel<128>, dim3((unsigned)p->n_rows), dim3(128), smem, st, a);
            else
                hipLaunchKernelGGL(beam_merge2_kernel<256>, dim3((unsigned)p->n_rows), dim3(256), smem, st, a);
            VL_LAUNCH_CHECK("beam merge kernel");
            if (prof) VL_HIP(hipEventRecord(ev[3 * at + 2], st));
        }
        BeamReport found;
        if (ahead) {
            rc = launch_next();
            if (rc < 0) return rc;
            const int waited = slot.wait((int)checked);
            if (waited < -1) VL_HIP((hipError_t)(-1 - waited));
            if (waited < 0) {
                vl_set_error("the progress check after iteration %lld was not reported", (long long)checked);
                return VL_ERR_HIP;
            }
            found = *slot.get();
            // the launch that has nothing left to do is waited for: the caller may use the workspace on another stream
            if ((!found.changed && !found.refused_at) || found.error) {
                VL_HIP(hipStreamSynchronize(st));
                slot.drained();
            }
        } else {
            // one copy brings the ring of progress flags and the three words behind it (they are neighbours in the
            // control block): this check's flag, the rows still using the sketch, the error flag
            struct {
                int changed[64];
                int sketch_rows, error, refused_at;
            } seen_by_host;
            static_assert(offsetof(BeamCtrl, refused_at) - offsetof(BeamCtrl, changed) == 66 * sizeof(int) &&
                              offsetof(BeamCtrl, error) - offsetof(BeamCtrl, changed) == 65 * sizeof(int) &&
                              offsetof(BeamCtrl, sketch_rows) - offsetof(BeamCtrl, changed) == 64 * sizeof(int),
                          "changed[64], sketch_rows, error, refused_at follow each other");
            VL_HIP(hipMemcpyAsync(&seen_by_host, &ctrl->changed[0], sizeof(seen_by_host), hipMemcpyDeviceToHost, st));
            VL_HIP(hipStreamSynchronize(st));
            slot.drained();
            found.changed = seen_by_host.changed[(checked / R) & 63];
            found.sketch_rows = seen_by_host.sketch_rows;
            found.error = seen_by_host.error;
            found.refused_at = seen_by_host.refused_at;
        }
        if (sketch_table) sketch_rows = found.sketch_rows;
        if (found.error) {
            vl_set_error("a row's visited list holds more ids than %lld iterations can have put there: the workspace "
                         "was overwritten while the loop ran - is it shared with a concurrent call?", (long long)checked);
            return VL_ERR_STATE;
        }
        if (prof) {
            for (int r = 0; r < launches; ++r) {
                float ms = 0;
                VL_HIP(hipEventElapsedTime(&ms, ev[3 * r], ev[3 * r + 1]));
                mine.expand_ms += ms;
                if (!use_fused) {
                    VL_HIP(hipEventElapsedTime(&ms, ev[3 * r + 1], ev[3 * r + 2]));
                    mine.merge_ms += ms;
                }
            }
            mine.expand_launches += launches;
            mine.merge_launches += launches;
        }
        if (table && found.refused_at) {
            // the launches from iteration refused_at on did nothing: the loop goes on from there without the table
            table = false;
            hipLaunchKernelGGL(beam_resume_kernel, dim3(1), dim3(64), 0, st, ctrl);
            VL_LAUNCH_CHECK("beam_resume_kernel");
            step.memo = l.memo_slots > 0 ? memo : nullptr;
            rc = make_ready(true);
            if (rc < 0) return rc;
            t = found.refused_at - 1;
            if (ahead) slot.forget();  // (a check may be made again)
            const bool checked_there = t == checked;
            checked = t;
            if (!checked_there) continue;
        }
        if (!found.changed) break;  // ann.py:90-91
        if (checked > t_limit) {
            vl_set_error("beam search still changing after %lld iterations (bound %lld): its workspace was "
                         "overwritten while it ran - is it shared with a concurrent call?",
                         (long long)checked, (long long)t_limit);
            return VL_ERR_STATE;
        }
    }
    if (prof) {
        unsigned long long ev_counts[kBeamStripes];
        VL_HIP(hipMemcpyAsync(ev_counts, ctrl->evals, sizeof(ev_counts), hipMemcpyDeviceToHost, st));
        VL_HIP(hipStreamSynchronize(st));
        for (int i = 0; i < kBeamStripes; ++i) mine.evals += (int64_t)ev_counts[i];
        VL_HIP(hipMemcpyAsync(ev_counts, ctrl->wanted, sizeof(ev_counts), hipMemcpyDeviceToHost, st));
        VL_HIP(hipStreamSynchronize(st));
        for (int i = 0; i < kBeamStripes; ++i) mine.wanted += (int64_t)ev_counts[i];
        VL_HIP(hipMemcpyAsync(ev_counts, ctrl->sketched, sizeof(ev_counts), hipMemcpyDeviceToHost, st));
        VL_HIP(hipStreamSynchronize(st));
        for (int i = 0; i < kBeamStripes; ++i) mine.sketched += (int64_t)ev_counts[i];
        std::lock_guard<std::mutex> hold(g_prof_mutex);
        g_prof.expand_ms += mine.expand_ms; g_prof.merge_ms += mine.merge_ms;
        g_prof.expand_launches += mine.expand_launches; g_prof.merge_launches += mine.merge_launches;
        g_prof.evals += mine.evals; g_prof.wanted += mine.wanted; g_prof.sketched += mine.sketched;
        g_prof.rows += p->n_rows;
        g_prof.iterations += checked;
    }
    return checked;
}

}  // namespace

VL_EXPORT int64_t vl_closest_vectors(const vl_beam_params *p, const float *queries, const float *vectors,
                                     const int32_t *beams, int32_t *q_ids, float *q_dists,
                                     const int32_t *exclude, void *workspace, int64_t workspace_bytes,
                                     void *stream) {
    BeamLayout l;
    int rc = beam_layout(p, &l);
    if (rc < 0) return rc;
    if (p->n_rows == 0) return 0;
    return beam_loop(p, l, queries, vectors, beams, q_ids, q_dists, exclude, workspace, workspace_bytes, 0, nullptr,
                     stream);
}

VL_EXPORT int64_t vl_closest_vectors_with_sketch(const vl_beam_params *p, const float *queries, const float *vectors,
                                                 const uint8_t *sketch, const int32_t *beams, int32_t *q_ids,
                                                 float *q_dists, const int32_t *exclude, void *workspace,
                                                 int64_t workspace_bytes, void *stream) {
    BeamLayout l;
    int rc = beam_layout(p, &l);
    if (rc < 0) return rc;
    VL_REQUIRE(!sketch || ((uintptr_t)sketch & 15) == 0, "the sketch table must be 16-byte aligned");
    if (p->n_rows == 0) return 0;
    return beam_loop(p, l, queries, vectors, beams, q_ids, q_dists, exclude, workspace, workspace_bytes, 0, nullptr,
                     stream, sketch);
}

// ---- the entry point that allocates nothing -------------------------------------------
// Its scratch memory is this array, part of the loaded code object: every GPU the library runs on holds
// its own copy until the process ends.  In host code the array's name is only a handle; the address the
// kernels are given comes from hipGetSymbolAddress, looked up once per device with that device current.
namespace {

static __device__ __align__(256) unsigned char scratch[VL_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
void *g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_mutex;

int scratch_of_current_device(void **out) {
    int dev = -1;
    VL_HIP(hipGetDevice(&dev));
    VL_REQUIRE(dev >= 0 && dev < kMaxDevices, "device index %d is out of range", dev);
    std::lock_guard<std::mutex> hold(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        VL_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        VL_REQUIRE(ptr != nullptr, "no device address for the static scratch array");
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return VL_OK;
}

}  // namespace

VL_EXPORT int vl_closest_vectors_noalloc(const vl_beam_params *p, const float *queries, const float *vectors,
                                         const int32_t *beams, int32_t *q_ids, float *q_dists,
                                         const int32_t *exclude, int64_t iterations, int32_t *status_out,
                                         void *stream) {
    BeamLayout l;
    int rc = beam_layout(p, &l, true);
    if (rc < 0) return rc;
    VL_REQUIRE(iterations >= 1 && iterations <= 65536, "iterations must be between 1 and 65536");
    VL_REQUIRE(status_out, "null pointer");
    VL_REQUIRE((p->flags & (VL_BEAM_TWO_LAUNCHES | VL_BEAM_SORT_MERGE)) == 0,
               "only the fused step runs without a caller's workspace");
    VL_REQUIRE(l.total <= (int64_t)VL_NOALLOC_SCRATCH_BYTES,
               "this batch needs %lld bytes of scratch memory, the static array holds %lld: use fewer rows per call "
               "(about %lld bytes per row) or vl_closest_vectors with a workspace",
               (long long)l.total, (long long)VL_NOALLOC_SCRATCH_BYTES,
               (long long)(l.VL * 8 + l.E * 4 + 8));
    void *ptr = nullptr;
    rc = scratch_of_current_device(&ptr);
    if (rc < 0) return rc;
    if (p->n_rows == 0) {
        // nothing to search: the loop ended after no iteration
        hipLaunchKernelGGL(beam_empty_status_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, status_out);
        VL_LAUNCH_CHECK("beam_empty_status_kernel");
        return VL_OK;
    }
    return (int)beam_loop(p, l, queries, vectors, beams, q_ids, q_dists, exclude, ptr, VL_NOALLOC_SCRATCH_BYTES,
                          iterations, status_out, stream);
}

// Profiling switch for vl_closest_vectors: when enabled every expand / merge
// launch is bracketed by HIP events on the caller's stream and the fetched
// candidate rows are counted.  out[0..7] = expand ms, merge ms, expand
// launches, merge launches, candidate rows fetched, query rows, iterations,
// candidate distances asked for (fetched + served by the per-row cache),
// out[8] = candidate rows looked at through the sketch, summed since the last
// reset.
VL_EXPORT int64_t vl_beam_launches(void) { return g_step_launches.load(std::memory_order_relaxed); }

VL_EXPORT int vl_beam_profile(int enable, int reset, double *out) {
    std::lock_guard<std::mutex> hold(g_prof_mutex);
    if (out) {
        out[0] = g_prof.expand_ms; out[1] = g_prof.merge_ms;
        out[2] = (double)g_prof.expand_launches; out[3] = (double)g_prof.merge_launches;
        out[4] = (double)g_prof.evals; out[5] = (double)g_prof.rows; out[6] = (double)g_prof.iterations;
        out[7] = (double)g_prof.wanted;
        out[8] = (double)g_prof.sketched;
    }
    if (reset) g_prof = BeamProfile();
    g_prof.enabled = enable;
    return VL_OK;
}
