// One row of the fused beam-search step (ann.py:68-88): pop the visit-queue heads, gather their neighbour lists,
// evaluate the candidates, insert them into the search queue and refill the visit queue, in one workgroup.
//
// The row's visited ids are an unordered list in memory (appended to) and a hash set in LDS while a workgroup has the
// row.  Every candidate claims its id in the same set, so one access tells a visited id, a later copy of an id within
// the iteration and a new candidate apart.  What the two queues keep is found without sorting: a survivor's place is its
// lower bound in the queue plus the number of smaller survivors, a queued key's place moves by the number of survivors
// below it.  (Lists kept sorted, Vt workgroup-wide minima and a bitonic sort of the survivors, which this replaces, took
// 7,700 + 3,400 + 3,500 of 40,000 cycles of a lone workgroup at 4,096 x 128, degree 32, and the searches of the visited
// list 3,000 more.)
#pragma once
#include "beam_ctrl.h"
#include "rowsort.h"
#include "dist_device.h"
#include "near_products.h"
#include "sketch_device.h"

constexpr int kMaxVisit = 64;  // parallel_visit_count handled by one wavefront

struct MergeArgs {
    BeamCtrl *ctrl;
    int iter;
    int readahead;
    int64_t n_rows;
    const int32_t *cand_ids;
    const float *cand_d;
    int m;
    int32_t *q_ids;
    float *q_d;
    int cap, L, Ps;
    const int32_t *excl;
    int excl_cols;
    int32_t *v_ids;
    float *v_d;
    int VL, Vt, Pv, Pc;
    int32_t *seen;
    int32_t *seen_count;
    int E;
    int32_t *row_quiet;  // per-query stop only (else null): iterations in a row that left the row's search queue unchanged
};

struct StepArgs {
    MergeArgs m;
    const float *queries;
    const float *vectors;
    const int32_t *beams;
    int64_t n_vectors;
    int dim, nchunks, width;
    uint32_t width_magic;  // floor(2^32 / width) + 1: slot / width == umulhi(slot, width_magic) for slot * width < 2^32
    uint64_t *memo;
    int memo_shift;
    int32_t *memo_rate;   // per row: share (x 256) of the candidates of iteration kMemoDecide that were cached; bit 16: the row uses the sketch
    int memo_min_rate;    // the cache stays in use only if that share is at least this (x 256)
    int count_evals;
    int l2;  // 0: cosine distance, 1: squared L2
    const uint8_t *sketch;     // 8-bit sketch of `vectors` (sketch_device.h), or null
    const uint8_t *sketch_tails;  // the table's second part: 8 bytes per vector
    int sketch_chunks;         // 16-byte chunks of data in a sketch row
    const uint8_t *rounded_queries;  // the call's query rows rounded for the sketch (sketch_device.h)
    int64_t rounded_query_bytes;
    const uint16_t *near_values;    // products of the call's queries and vectors (near_products.h), instead of the sketch's rows; or null
    const uint32_t *near_columns;   // what is known of the vector of a column
    const NearQuery *near_queries;
    int64_t near_pitch;
    int hash_slots;      // slots of the LDS hash set (row_hash_slots)
    int window;          // > 0: iterations m.iter ... m.iter + window - 1 in this launch
    BeamReport *report;  // pinned host memory that hears of the progress checks, or null
};

// Slots of a row's hash set, a multiple of 4 (it is cleared 16 bytes at a time).  The fewest: three quarters of them taken
// by visited ids and candidates; outside windows also room for m keys.  The most that are any use: a quarter taken.
__host__ __device__ inline int row_hash_slots(int64_t visited, int64_t m, bool window) {
    int64_t slots = (visited + m) * 4 / 3 + 7;
    if (!window && slots < 2 * m + 3) slots = 2 * m + 3;
    return (int)(slots & ~3ll);
}
__host__ __device__ inline int row_hash_slots_most(int64_t visited, int64_t m) { return (int)(4 * (visited + m)); }

// LDS of a row's workgroup, in bytes from the start of its dynamic LDS.
//   keys   m keys: the survivors; before that the sketched candidates' upper bounds
//   cand   m ids and m distances; after the survivors have been picked m keys, the new ones of the search queue
//   qa, vq the queues as keys (all VL slots of the visit queue, the popped heads first); a window keeps two of each
//   set    the hash set
//   fresh  m keys, the new ones of the visit queue: over the hash set, which is done with by then except in a window
struct RowLayout {
    int cand, qa, vq, set, fresh, slot, exl, flags, bytes;
};
__host__ __device__ inline RowLayout row_layout(int m, int L, int VL, int hash_slots, int excl_cols, bool window) {
    RowLayout o;
    const int m2 = (m + 1) & ~1, copies = window ? 2 : 1;
    o.cand = 8 * m2;
    o.qa = o.cand + 8 * m2;
    o.vq = o.qa + 8 * copies * L;
    o.set = (o.vq + 8 * copies * VL + 15) & ~15;
    int end = o.set + 4 * hash_slots;
    o.fresh = o.set;
    if (window) {
        o.fresh = (end + 7) & ~7;
        end = o.fresh + 8 * m;
    }
    o.exl = end;
    end += 4 * excl_cols;
    o.slot = end;  // window only: 16 bits per candidate, where it sits in the hash set
    if (window) end += 2 * m2;
    o.flags = end;
    o.bytes = end + m;
    return o;
}

// Raise the batch-wide running maximum *slot to at least cnt.  Same-address
// atomics from thousands of workgroups serialise in L2 and were the most
// expensive part of the merge step, so they are kept for the rare case only:
// a row that is at the largest fill any row can have (bound) publishes it with
// a plain store - every such writer stores the same value and no atomicMax of a
// smaller value can lower it - and any row skips the update when a late read
// shows the slot is already there.
__device__ inline void raise_running_max(int *slot, int cnt, int bound) {
    if (__hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= cnt) return;
    if (cnt >= bound) __hip_atomic_store(slot, cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else atomicMax(slot, cnt);
}

// A candidate's upper bound (a cosine distance, in [0, 1]) and its slot in one 32-bit key, smallest bound first:
// the bound to 19 bits, rounded down, then the slot (a row has at most kMaxCandidates candidate slots: more would
// not fit the LDS).  Only used to choose which candidates to look at first - any choice is a valid one there - so
// the rounding costs nothing but a slightly different pick among near-equal bounds.  Never 0xFFFFFFFF.
constexpr int kMaxCandidates = 8192;
__device__ __forceinline__ uint32_t bound_slot_key(float hi, int slot) {
    return ((uint32_t)(hi * 524286.0f) << 13) | (uint32_t)slot;
}

// A probe of the distance cache is a random 8-byte read and every evaluated distance a random 8-byte
// write - a memory sector each, and one more round trip before the candidate rows can be asked for - so
// the cache only pays when enough probes hit; how many depends on the row size (short rows are cheap to
// fetch again).  Each row therefore decides for itself: it uses the cache during its first kMemoDecide - 1
// iterations, measures the share of hits in iteration kMemoDecide, and leaves the cache alone for the rest
// of the call if that share is below the break-even share.  A hit returns the bits that would be computed
// again, so the decision never changes a result.  (Where rows ask for so many candidates that they meet most vectors
// again, meets_again in beam.hip, the break-even share is 0: the cache stays in use.)
constexpr int kMemoDecide = 9;

// Elements of a row that one thread brings in at the start of the fused step and keeps in registers until
// the workgroup's other reads have been issued: search queue, visit queue, visited list.  Longer rows load
// their remainder the slow way (read, wait, store): a visited list of more than 512 ids in 128 threads has one, which rows of
// a degree of 35 and more reach late in a call (960 ids at degree 64), and a queue of more than 256 slots.
constexpr int kPreQ = 2, kPreV = 2, kPreS = 4;

// Takes id's place in an open-addressed set (-1: empty).  False: the id is there already.  The places tried are those of a
// sequence that runs through all 32-bit values (a full-period congruence), so an empty one is met.  64 ids wait for the
// longest of their searches, which is why the set is kept as empty as LDS allows: 256 queries at 4,096 x 128 take 1,462 us
// with three quarters of the set taken and the next place tried after a taken one, 1,004 us with a quarter of it taken.
__device__ __forceinline__ bool set_claim(int32_t *set, uint32_t slots, int32_t id, uint32_t *at) {
    uint32_t x = (uint32_t)id * 2654435761u;
    for (;;) {
        const uint32_t h = __umulhi(x, slots);
        const int32_t there = atomicCAS(&set[h], -1, id);
        if (there == -1) {
            *at = h;
            return true;
        }
        if (there == id) return false;
        x = x * 1664525u + 1013904223u;
    }
}

// Smallest value of each row of 16 lanes, in all of them.
__device__ __forceinline__ uint32_t row16_min_u32(uint32_t x) {
    uint32_t y;
    y = __builtin_amdgcn_update_dpp(x, x, 0x128, 0xf, 0xf, false); x = y < x ? y : x;  // row_ror:8
    y = __builtin_amdgcn_update_dpp(x, x, 0x124, 0xf, 0xf, false); x = y < x ? y : x;  // row_ror:4
    y = __builtin_amdgcn_update_dpp(x, x, 0x122, 0xf, 0xf, false); x = y < x ? y : x;  // row_ror:2
    y = __builtin_amdgcn_update_dpp(x, x, 0x121, 0xf, 0xf, false); x = y < x ? y : x;  // row_ror:1
    return x;
}

// red[0 .. N): N values in LDS.  The lane's own (lane mod N) and its rank among them, equal ones by place.
template <int N>
__device__ __forceinline__ uint32_t rank_among(const uint32_t *red, int *rank) {
    const int own = threadIdx.x & (N - 1);
    const uint32_t mine = red[own];
    int r = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const uint32_t other = red[i];
        r += other < mine || (other == mine && i < own);
    }
    *rank = r;
    return mine;
}

// A count that all lanes of the wavefront have read from LDS, in a scalar register if SCALAR: loops up to it have no lane masks.
template <bool SCALAR>
__device__ __forceinline__ int same_in_all(int x) {
    return SCALAR ? __builtin_amdgcn_readfirstlane(x) : x;
}

// keys: n of them in LDS (n the same in all lanes); places past the last are not read.  N reads are on their way at a time:
// one after the other, a key costs the latency of LDS.
template <int N>
__device__ __forceinline__ int count_below(const uint64_t *keys, int n, uint64_t k) {
    int c = 0, i = 0;
    for (; i + N <= n; i += N) {
        uint64_t x[N];
#pragma unroll
        for (int j = 0; j < N; ++j) x[j] = keys[i + j];
#pragma unroll
        for (int j = 0; j < N; ++j) c += x[j] < k;
    }
    if (N > 1 && i < n) {
        uint64_t x[N];
#pragma unroll
        for (int j = 0; j < N - 1; ++j) x[j] = keys[i + j < n ? i + j : n - 1];
#pragma unroll
        for (int j = 0; j < N - 1; ++j) c += i + j < n && x[j] < k;
    }
    return c;
}

// Lower bounds of k in two sorted arrays at once: the steps of the two searches wait for LDS together.
__device__ __forceinline__ void two_lower_bounds(const uint64_t *a, int na, int *in_a, const uint64_t *b, int nb, int *in_b,
                                                 int top, uint64_t k) {
    int x = 0, y = 0;
    for (int step = top; step > 0; step >>= 1) {  // top: the largest power of two not above the longer one's length
        const int i = x + step, j = y + step;  // (selects, no branches: those cost more than the reads past the end they save)
        const uint64_t in_a = a[min(i, na) - 1], in_b = b[min(j, nb) - 1];
        x = ((i <= na) & (in_a < k)) ? i : x;
        y = ((j <= nb) & (in_b < k)) ? j : y;
    }
    *in_a = x;
    *in_b = y;
}

// SCPL > 0: the kernel can look at candidates through the sketch first (SCPL chunks per lane, SLPR lanes
// per sketch row, SU loads in flight).  A row that does so gets bounds for the candidates the distance cache
// does not know from a quarter of the bytes, then exact distances for the few whose lower bound is not above
// every threshold that decides what the queues keep; it stops doing so when most of them turn out to
// need their exact distance (bit 16 of its word in memo_rate: set at the start of the call, cleared then).
//
// WINDOW: the launch takes the row through iterations m.iter ... m.iter + window - 1 with its queues and visited ids in
// LDS.  While parallel_visit_count * t <= E (the visited list's width) no row's visited list can be full at iteration t,
// so every row records all the ids it pops (utils.py:73-75 with room for them in every row) and nothing a row does
// between two progress checks depends on another row of the batch; the only batch-wide facts, the progress flag of the
// checking iteration (ann.py:90-91) and the largest fill after the last of them, are written once.  Such a launch starts
// right after a progress check (m.iter = k * readahead + 1, window = readahead).
//
// NEAR: bounds come from the call's table of products (near_products.h), one look each.  They are not worth the cache, which
// keeps exact distances only.
template <int CPL, int LPR, int U, RowForm FORM, int THREADS, int SCPL = 0, int SLPR = 64, int SU = 1, bool WINDOW = false, bool NEAR = false>
__device__ __forceinline__ void beam_row(const StepArgs &s) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int kRows16 = THREADS / 16;
    // Queue keys read at a time when places are counted: eight for several iterations of rows of up to 384 elements (256
    // queries at 4,096 x 128 1,006 -> 969 us, 10,000 at 1M x 128 2,063 -> 2,017, a build of 6,007 x 384 17.5 -> 17.0 ms).
    // Longer rows hide the latency behind each other's loads (1,000 queries at 100,003 x 1,536 1,239 us with one, 1,267 with
    // eight; 10,000 at 1M x 768 3,513 and 3,527), and the kernels of one iteration have no registers left for it (a build of
    // 20,011 x 768 133.1 and 133.7 ms).
    constexpr bool kShortRows = WINDOW && SCPL == 0 && CPL * LPR <= 96;
    constexpr int kAtOnce = kShortRows ? 8 : 1;
    // Whether a wavefront's sums become distances together (listed_distances).  Of aligned rows those of 129 to 256 columns: 64
    // lanes bring one row a load, and eight loads wait for eight stores.  Away and together: batches of a first loop at 100,000 x
    // 200 65.4 -> 63.9 ms (degree 64) and 16.2 -> 15.4 (32), builds of 8,000 x 200 16.2 -> 15.2, 300 / 1,000 / 10,000 queries at
    // 20,000 x 200 2,950 -> 2,694, 3,194 -> 2,738 (degree 32) and 33,314 -> 32,890 us; clusters of 977 at 60,000 x 256 6,393 -> 6,508.
    constexpr bool kSums = FORM == kRowUnalignedSums || (FORM == kRowAligned && SCPL == 0 && CPL == 1 && LPR == 64);
    // Sets of 64 candidates of a wavefront whose neighbour ids and cache probes are on their way at a time.  (The kernels with
    // the sketch, which wait on bytes, spill registers with two: a batch of the first loop at 1M x 768 141.0 and 143.1 ms.  With
    // the table of products, whose looks are on their way along with them, two are the sooner: 59.9 -> 59.2, 500,000 x 1,024 61.0 ->
    // 57.6, 1M x 384 37.8 -> 35.9.)
    constexpr int kAhead = SCPL > 0 && !NEAR ? 1 : 2;
    // Where the ids to visit are read from: the heads of the visit queue, and in the kernels with the sketch a copy of their
    // own, which those need to be as fast (a batch of the first loop at 1M x 768 141.3 ms without it, 139.9 with it).
    constexpr bool kOwnHeads = SCPL > 0 && !NEAR;
    __shared__ int32_t visit_s[kOwnHeads ? kMaxVisit : 1];
    __shared__ uint32_t red[kRows16];
    __shared__ int n_ex_s;                  // exclusion ids before the row's first empty one
    __shared__ int n_keys_s, n_search_s, n_fresh_s, n_miss_s, changed_s, n_new_s, probe_hits_s, probe_asked_s, quiet_s, word_s;
    __shared__ __align__(8) uint8_t order_s[THREADS];  // lists of candidate lanes (wave_sketch, wave_distances_lds), 64 bytes per wavefront

    const MergeArgs &a = s.m;
    BeamCtrl *c = a.ctrl;
    const int t0 = a.iter;
    int tid = threadIdx.x;
    int lane = tid & (kWave - 1);
    int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int64_t row = blockIdx.x;
    const int nva = a.VL - a.Vt;
    // ---- every read that depends on nothing else goes out first: loop state, the row's counters, the ids
    // to visit, both queues, the visited list, the exclusions.  A round trip to memory costs more than
    // anything this workgroup computes, so the number of dependent round trips is what it pays for: this
    // one, then the neighbour lists of the visited ids, the cache probes, the candidate rows.
    int32_t *vi = a.v_ids + row * a.VL;
    float *vd = a.v_d + row * a.VL;
    int32_t *qi = a.q_ids + row * a.cap;
    float *qd = a.q_d + row * a.cap;
    int32_t *srow = a.seen + row * a.E;
    const int seen_bound = min(a.E, a.Vt * (t0 - 1));  // the fill is at most Vt ids per earlier iteration
    const int32_t my_visit = tid < a.Vt ? vi[tid] : VL_MAXINT;
    int cnt = a.seen_count[row];
    const int first0 = WINDOW ? 0 : c->first[t0 % 3];  // first visited-list column that is free in every row
    const int quiet0 = a.row_quiet ? a.row_quiet[row] : 0;
    int memo_word = s.memo_rate[row];
    int32_t pq_i[kPreQ], pv_i[kPreV], ps[kPreS];
    float pq_d[kPreQ], pv_d[kPreV];
#pragma unroll
    for (int j = 0; j < kPreQ; ++j) {
        const int i = tid + j * THREADS;
        pq_i[j] = i < a.L ? qi[i] : VL_MAXINT;
        pq_d[j] = i < a.L ? qd[i] : VL_MAXFLOAT;
    }
#pragma unroll
    for (int j = 0; j < kPreV; ++j) {
        const int i = tid + j * THREADS;
        pv_i[j] = i < nva ? vi[a.Vt + i] : VL_MAXINT;
        pv_d[j] = i < nva ? vd[a.Vt + i] : VL_MAXFLOAT;
    }
#pragma unroll
    for (int j = 0; j < kPreS; ++j) {
        const int i = tid + j * THREADS;
        ps[j] = i < seen_bound ? srow[i] : VL_MAXINT;
    }
    int32_t my_excl = VL_MAXINT;
    if (a.excl && tid < a.excl_cols) my_excl = a.excl[row * a.excl_cols + tid];

    // (WINDOW: the visited lists cannot be full in these iterations; the slots of `first` are not read, because rows of
    // this very launch that finish early write the one the next launch reads)
    const int gate = beam_gate(c, t0, a.readahead, a.E, blockIdx.x == 0 && tid == 0, s.report, !WINDOW);
    if (gate == 2) return;
    if (!beam_row_state_ok(c, cnt, seen_bound, tid == 0)) return;
    const int iterations = WINDOW ? s.window : 1;
    int *const first_after = &c->first[(t0 + iterations) % 3];  // what the launch of iteration t0 + iterations reads
    const int bound_after = min(a.E, a.Vt * (t0 + iterations - 1));
    if (gate == 1 || (a.row_quiet && quiet0 >= a.readahead)) {
        // the visit queue is no longer fed (every candidate of this iteration is empty), or this row has
        // stopped on its own: nothing changes, only the running maximum is kept current
        if (tid == 0) raise_running_max(first_after, cnt, bound_after);
        return;
    }
    const uint32_t slots = (uint32_t)s.hash_slots;
    const RowLayout at = row_layout(a.m, a.L, a.VL, s.hash_slots, a.excl_cols, WINDOW);
    uint64_t *const keys = reinterpret_cast<uint64_t *>(smem);
    uint16_t *const missed = reinterpret_cast<uint16_t *>(smem);  // candidate slots to fetch (before there are keys)
    float *const le = reinterpret_cast<float *>(smem);  // upper bounds of sketched candidates (keys are picked later)
    int32_t *const li = reinterpret_cast<int32_t *>(smem + at.cand);
    float *const ld = reinterpret_cast<float *>(li + a.m);
    uint64_t *const to_search = reinterpret_cast<uint64_t *>(smem + at.cand);
    uint64_t *const to_visit = reinterpret_cast<uint64_t *>(smem + at.fresh);
    int32_t *const set = reinterpret_cast<int32_t *>(smem + at.set);
    int32_t *const exl = reinterpret_cast<int32_t *>(smem + at.exl);
    uint16_t *const set_slot = reinterpret_cast<uint16_t *>(smem + at.slot);
    uint8_t *const flags = smem + at.flags;
    uint64_t *qa = reinterpret_cast<uint64_t *>(smem + at.qa);
    uint64_t *vq = reinterpret_cast<uint64_t *>(smem + at.vq);
    uint64_t *qa_next = qa + a.L, *vq_next = vq + a.VL;  // WINDOW only
    const float *q_row = s.queries + row * s.dim;
    uint64_t *const memo_table = s.memo ? s.memo + ((uint64_t)row << (32 - s.memo_shift)) : nullptr;
    uint8_t *const order = order_s + wave * kWave;

    for (int i = tid; i < (int)(slots >> 2); i += THREADS) reinterpret_cast<int4 *>(set)[i] = make_int4(-1, -1, -1, -1);
    if (tid < a.Vt) {  // the ids popped in the first iteration
        if constexpr (kOwnHeads) visit_s[tid] = my_visit;
        else vq[tid] = vl_make_key(my_visit, VL_MAXFLOAT);
    }
    if (tid == 0) {
        n_ex_s = a.excl ? a.excl_cols : 0;
        quiet_s = quiet0;
    }
    __syncthreads();

    auto popped = [&](int i) -> int32_t {  // queue.py:87-95: the heads are popped
        if constexpr (kOwnHeads) return visit_s[i];
        else return vl_key_id(vq[i]);
    };
    // candidate id of a slot: the neighbour list of a visited node (ann.py:69-73)
    auto resolve = [&](int slot) -> int32_t {
        int32_t id = VL_MAXINT;
        if (slot < a.m) {
            int sidx = s.width == 1 ? slot : (int)__umulhi((uint32_t)slot, s.width_magic), k = slot - sidx * s.width;
            const int32_t node = popped(sidx);
            if (node != VL_MAXINT && (uint32_t)node < (uint64_t)s.n_vectors) id = s.beams[(int64_t)node * s.width + k];
        }
        return id;
    };
    // (those of a wavefront's first kAhead sets of candidates are asked for ahead of everything else)
    int32_t near[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) near[j] = wave * kWave + j * THREADS < a.m ? resolve(tid + j * THREADS) : VL_MAXINT;
    // The row's own state, read at the top, goes to LDS now that the first neighbour lists are on their
    // way.  (Outside the loops below on purpose: inside, its addresses would be kept in registers across
    // the distance code.)
    {
        uint32_t h;
#pragma unroll
        for (int j = 0; j < kPreQ; ++j) {
            const int i = tid + j * THREADS;
            if (i < a.L) qa[i] = vl_make_key(pq_i[j], pq_d[j]);
        }
#pragma unroll
        for (int j = 0; j < kPreV; ++j) {
            const int i = tid + j * THREADS;
            if (i < nva) vq[a.Vt + i] = vl_make_key(pv_i[j], pv_d[j]);
        }
#pragma unroll
        for (int j = 0; j < kPreS; ++j)
            if (tid + j * THREADS < cnt) set_claim(set, slots, ps[j], &h);
        if (a.excl && tid < a.excl_cols) {
            exl[tid] = my_excl;
            if (my_excl == VL_MAXINT) atomicMin(&n_ex_s, tid);
        }
        for (int i = tid + kPreQ * THREADS; i < a.L; i += THREADS) qa[i] = vl_make_key(qi[i], qd[i]);
        for (int i = tid + kPreV * THREADS; i < nva; i += THREADS) vq[a.Vt + i] = vl_make_key(vi[a.Vt + i], vd[a.Vt + i]);
        for (int i = tid + kPreS * THREADS; i < cnt; i += THREADS) set_claim(set, slots, srow[i], &h);
        for (int i = tid + THREADS; i < a.excl_cols; i += THREADS) {
            int32_t e = a.excl[row * a.excl_cols + i];
            exl[i] = e;
            if (e == VL_MAXINT) atomicMin(&n_ex_s, i);
        }
    }
    bool queue_moved = false;  // WINDOW: the search queue in LDS is not the one in memory any more

    for (int w = 0; w < iterations; ++w) {
        const int t = t0 + w;
        if constexpr (WINDOW) {
            // what follows from these is worked out in every iteration again: kept across iterations, the lane masks,
            // addresses and query row took 30 registers more than the one-iteration kernel has
            asm volatile("" : "+v"(tid), "+s"(q_row));
            lane = tid & (kWave - 1);
            wave = __builtin_amdgcn_readfirstlane(tid / kWave);
        }
        if (WINDOW && w > 0) {
            if constexpr (kOwnHeads) {
                if (tid < a.Vt) visit_s[tid] = vl_key_id(vq[tid]);
                __syncthreads();
            }
#pragma unroll
            for (int j = 0; j < kAhead; ++j) near[j] = wave * kWave + j * THREADS < a.m ? resolve(tid + j * THREADS) : VL_MAXINT;
            memo_word = word_s;
        }
        const int first = WINDOW ? a.Vt * (t - 1) : first0;
        const bool seen_full = first >= a.E;  // add_new_to_seen_ returns None now (utils.py:68-69)
        const bool checking = (t % a.readahead) == 0;
        const int memo_rate = memo_word & 0xffff;
        const bool resample = memo_table && t == kMemoDecide;
        uint64_t *const memo_row = memo_table && memo_rate >= s.memo_min_rate ? memo_table : nullptr;
        const bool probing = memo_row && t > 1;  // nothing is cached before the first iteration, whose candidates are distinct
        // (not in the first iteration: the visit queue starts with empty slots, so everything unvisited is kept and
        // would be fetched anyway)
        bool sketching = false;
        if constexpr (SCPL > 0) sketching = s.sketch != nullptr && (memo_word >> 16) != 0 && t > 1;
        if (w == 0) __syncthreads();  // the queues and the visited ids are in LDS

        // ---- add_new_to_seen_ (utils.py:61-82): the popped ids that still have room become visited ----
        if (tid < kWave) {
            const int n_add = seen_full ? 0 : min(min(a.E - first, a.Vt), a.E - cnt);  // utils.py:73-75 (cnt <= first)
            const int32_t x = tid < n_add ? popped(tid) : VL_MAXINT;
            uint32_t h;
            const bool fresh = x != VL_MAXINT && set_claim(set, slots, x, &h);
            const uint64_t all = __ballot(fresh);
            const int n_new = __popcll(all);
            if (fresh) srow[cnt + __popcll(all & ((1ull << lane) - 1))] = x;
            if (tid == 0) {
                if (n_new) a.seen_count[row] = cnt + n_new;
                if (!WINDOW) raise_running_max(first_after, cnt + n_new, bound_after);
                n_new_s = n_new;
                n_keys_s = 0;
                n_search_s = 0;
                n_fresh_s = 0;
                n_miss_s = 0;
                changed_s = 0;
                probe_hits_s = 0;
                probe_asked_s = 0;
                word_s = memo_word;
            }
        }
        __syncthreads();

        // ---- expand: ann.py:69-73 ----
        int n_wanted = 0, n_fetched = 0, n_sketched = 0;  // counts of this wavefront
        // Two kinds of candidate become the empty pair here, before a probe or a row is spent on them.  One that the
        // visited list holds once this iteration has updated it can change neither queue: the visit queue excludes it
        // (ann.py:85-88), and the search queue met it with this very distance when it was first a candidate (every
        // visited id came out of the visit queue, which is fed from the search queue's heads and then with the
        // candidates the search queue is offered in the same iteration, ann.py:75-88), so it either still sits there or
        // lies beyond its last slot, which only ever moves down.  And later copies of an id: the neighbour lists of the
        // nodes visited in one iteration share ids; the reference evaluates every copy (kernels.py:238-255) and drops
        // all but one when the queues are sorted (kernels.py:314-349); copies carry the same distance.
        // A row without the sketch asks its cache for the others right away and lists the candidates to fetch.
        // With the table of products it gets their bounds, all of a set's looks on their way at a time.
        NearQuery nq;
        if constexpr (NEAR)
            if (sketching) nq = s.near_queries[row];
        for (int c0 = wave * kWave; c0 < a.m; c0 += kAhead * THREADS) {
            int32_t id[kAhead];
            bool ok[kAhead];
            uint64_t entry[kAhead];
            uint32_t value[kAhead], of_column[kAhead];
#pragma unroll
            for (int j = 0; j < kAhead; ++j) {
                const int slot = c0 + j * THREADS + lane;
                ok[j] = false;
                if (c0 + j * THREADS >= a.m) continue;  // uniform
                id[j] = c0 == wave * kWave ? near[j] : resolve(slot);
                ok[j] = slot < a.m && id[j] != VL_MAXINT && id[j] >= 0 && (int64_t)id[j] < s.n_vectors;
                if (s.count_evals || resample) n_wanted += __popcll(__ballot(ok[j]));
                uint32_t h = 0xffff;
                if (ok[j]) ok[j] = set_claim(set, slots, id[j], &h);
                if (slot < a.m) {
                    li[slot] = ok[j] ? id[j] : VL_MAXINT;
                    if (!ok[j]) ld[slot] = VL_MAXFLOAT;
                    if constexpr (WINDOW) set_slot[slot] = (uint16_t)(ok[j] ? h : 0xffffu);
                }
                if (!sketching && probing && ok[j]) entry[j] = memo_load(memo_row, s.memo_shift, id[j]);
                if constexpr (NEAR) {
                    if (sketching && ok[j]) {
                        const uint32_t column = PairColumns(s.n_vectors).of((uint32_t)id[j]);
                        value[j] = s.near_values[row * s.near_pitch + column];
                        of_column[j] = s.near_columns[column];
                    }
                }
            }
            if constexpr (NEAR) {
#pragma unroll
                for (int j = 0; j < kAhead; ++j) {
                    const int slot = c0 + j * THREADS + lane;
                    if (!sketching || slot >= a.m) continue;
                    flags[slot] = 0;
                    if (ok[j]) near_bounds(value[j], of_column[j], nq, ld + slot, le + slot);
                }
            }
            if (sketching) continue;
#pragma unroll
            for (int j = 0; j < kAhead; ++j) {
                const int slot = c0 + j * THREADS + lane;
                if (probing && ok[j] && (int32_t)(uint32_t)entry[j] == id[j]) {
                    ld[slot] = __builtin_bit_cast(float, (uint32_t)(entry[j] >> 32));
                    ok[j] = false;
                }
                const uint64_t all = __ballot(ok[j]);
                if (all == 0) continue;
                if (s.count_evals || resample) n_fetched += __popcll(all);
                int base = 0;
                if (lane == 0) base = atomicAdd(&n_miss_s, __popcll(all));
                base = __builtin_amdgcn_readfirstlane(base);
                if (ok[j]) missed[base + __popcll(all & ((1ull << lane) - 1))] = (uint16_t)slot;
            }
        }
        if constexpr (SCPL > 0 && !NEAR) {
            if (sketching) {
                SketchQuery<SCPL> sq;
                sketch_query_load<SCPL, SLPR>(sq, s.rounded_queries + row * s.rounded_query_bytes, s.sketch_chunks);
                for (int c0 = wave * kWave; c0 < a.m; c0 += THREADS) {
                    const int slot = c0 + lane;
                    const bool has = slot < a.m;
                    const int32_t id = has ? li[slot] : VL_MAXINT;
                    bool ok = id != VL_MAXINT;
                    if (has) flags[slot] = 0;
                    // The cache serves two kinds of repeats: a candidate evaluated exactly before comes back with its
                    // distance, one that was only bounded comes back with its bounds (dist_device.h) - either way
                    // nothing is fetched for it now.
                    if (memo_row && ok) {
                        const uint64_t e = memo_load(memo_row, s.memo_shift, id);
                        if ((int32_t)((uint32_t)e & ~kMemoBounds) == id) {
                            if ((uint32_t)e & kMemoBounds) {
                                ld[slot] = memo_bound_lo(e);
                                le[slot] = memo_bound_hi(e);
                            } else {
                                const float d = __builtin_bit_cast(float, (uint32_t)(e >> 32));
                                ld[slot] = d;
                                le[slot] = d;
                                flags[slot] = 16;  // exact already
                            }
                            ok = false;
                        }
                    }
                    if (s.count_evals || resample) n_sketched += __popcll(__ballot(ok));
                    wave_sketch<SCPL, SLPR, SU>(sq, s.sketch, s.sketch_tails, s.sketch_chunks, id, ok, ld + c0, le + c0,
                                                order, memo_row, s.memo_shift);
                }
                n_fetched = n_sketched;  // for the share of cache hits: what the cache did not answer
            }
        }
        if (!sketching) {
            __syncthreads();
            // (a scalar count: the loops up to it have no lane masks)
            const int n_miss = __builtin_amdgcn_readfirstlane(n_miss_s);
            if constexpr (FORM == kRowScalar) {
                for (int i = wave; i < n_miss; i += THREADS / kWave) {
                    const int slot = __builtin_amdgcn_readfirstlane(missed[i]);
                    wave_distances_generic(q_row, s.vectors, s.dim, s.nchunks, li[slot], lane == 0, ld + slot, memo_row,
                                           s.memo_shift, s.l2 != 0);
                }
            } else {
                listed_distances<CPL, LPR, U, THREADS / kWave, FORM != kRowAligned, kSums>(
                    q_row, s.vectors, s.dim, s.nchunks, li, missed, n_miss, wave, ld, memo_row, s.memo_shift, s.l2 != 0);
            }
        }
        const int stripe = (int)((blockIdx.x * (THREADS / kWave) + wave) & (kBeamStripes - 1));
        if (s.count_evals && lane == 0) {
            if (n_wanted) atomicAdd(&c->wanted[stripe], (unsigned long long)n_wanted);
            if (n_fetched && !sketching) atomicAdd(&c->evals[stripe], (unsigned long long)n_fetched);
            if (n_sketched) atomicAdd(&c->sketched[stripe], (unsigned long long)n_sketched);
        }
        if (resample && lane == 0) {
            atomicAdd(&probe_asked_s, n_wanted);
            atomicAdd(&probe_hits_s, n_wanted - n_fetched);
        }
        __syncthreads();
        if (resample && tid == 0) {
            const int word = (probe_asked_s > 0 ? (probe_hits_s * 256) / probe_asked_s : 256) | (memo_word & (1 << 16));
            s.memo_rate[row] = word;
            word_s = word;
        }
        const int n_ex = same_in_all<kShortRows>(n_ex_s);
        const uint64_t *const va = vq + a.Vt;
        const uint64_t ws = qa[a.L - 1];                       // the search queue's last slot
        const uint64_t wv = nva > 0 ? va[nva - 1] : 0ull;       // the visit queue's last live slot

        if constexpr (SCPL > 0) {
            // A sketched row knows every candidate distance only as lo <= d <= hi (ld holds lo, le holds hi).
            // What the queues keep of the candidates (all unvisited): keys below ws, keys below wv, and the Vt smallest
            // keys above wv.  Take any Vt candidates that are certainly above wv (lo > wv) - the smallest hi of 16-lane
            // groups, likely winners - evaluate them, and let tv be the
            // largest of their distances: Vt candidates are then known to be at most tv, so a candidate with
            // lo > tv is not one of the Vt smallest.  Hence a candidate whose lo is above ws, wv and tv cannot enter
            // either queue and is dropped; all others are
            // evaluated exactly, by the same code and in the same order as an unsketched row's, in two rounds
            // (the second one needs tv).  Comparisons are written so that a NaN bound counts as "evaluate".
            if (sketching) {  // uniform over the workgroup
                const float ws_d = vl_key_dist(ws);
                const float wv_d = nva > 0 ? vl_key_dist(wv) : -1.0f;
                uint32_t mine = 0xFFFFFFFFu;
                for (int i = tid; i < a.m; i += THREADS) {
                    uint8_t f = flags[i] & 16;  // set above for a distance that came from the cache
                    if (li[i] != VL_MAXINT) {
                        const float lo = ld[i];
                        bool need = !(lo > ws_d);
                        if (!seen_full) {
                            if (!(lo > wv_d)) need = true;
                            else {
                                f |= 2;  // certainly above the visit queue's last live slot
                                const uint32_t k = bound_slot_key(le[i], i);
                                mine = k < mine ? k : mine;
                            }
                        }
                        if (need) f |= 4;
                    }
                    flags[i] = f;
                }
                mine = row16_min_u32(mine);
                if ((lane & 15) == 0) red[tid >> 4] = mine;
                __syncthreads();
                // bit 8: one of the Vt (fewer groups than that have one: every candidate above wv is evaluated)
                bool all_rest = true;
                if (!seen_full) {
                    int rank;
                    const uint32_t x = rank_among<kRows16>(red, &rank);
                    const uint64_t chosen = __ballot(lane < kRows16 && rank < a.Vt && x != 0xFFFFFFFFu);
                    all_rest = __popcll(chosen) < a.Vt;
                    if (wave == 0 && ((chosen >> lane) & 1) && !all_rest) flags[x & (kMaxCandidates - 1)] |= 8;
                }
                __syncthreads();
                all_rest = __builtin_amdgcn_readfirstlane(all_rest) != 0;  // (a barrier below depends on it)
                int n_exact = 0, n_real = 0;
                // first round: everything below a queue's last slot, and those Vt candidates
                for (int c0 = wave * kWave; c0 < a.m; c0 += THREADS) {
                    const int slot = c0 + lane;
                    const bool has = slot < a.m;
                    const int32_t cid = has ? li[slot] : VL_MAXINT;
                    const uint8_t f = has ? flags[slot] : 0;
                    const bool ok = ((f & (4 | 8)) || (all_rest && (f & 2))) && !(f & 16);
                    if (ok) flags[slot] = f | 16;  // its distance is exact from here on
                    n_exact += __popcll(__ballot(ok));
                    n_real += __popcll(__ballot(cid != VL_MAXINT && !(f & 16)));  // candidates known by bounds only
                    wave_distances_lds<CPL, LPR, U>(q_row, s.vectors, s.dim, s.nchunks, cid, ok, ld + c0, order, memo_row,
                                                    s.memo_shift);
                }
                // tv: the largest exact distance of those Vt candidates.  Vt unvisited candidates above wv
                // are at most tv, so a candidate whose lower bound is above tv is not one of the Vt smallest.
                float tv = -1.0f;
                if (!seen_full && !all_rest) {
                    uint32_t least = 0xFFFFFFFFu;  // (no distance has the key 0)
                    for (int i = tid; i < a.m; i += THREADS)
                        if (flags[i] & 8) {
                            const uint32_t k = ~vl_float_key(ld[i]);
                            least = k < least ? k : least;
                        }
                    least = row16_min_u32(least);
                    if ((lane & 15) == 0) red[tid >> 4] = least;  // (every thread has read the group minima)
                    __syncthreads();
                    int rank;
                    const uint32_t x = rank_among<kRows16>(red, &rank);
                    const uint32_t top = (uint32_t)__builtin_amdgcn_readlane((int)x, __builtin_ctzll(__ballot(rank == 0)));
                    tv = top == 0xFFFFFFFFu ? -1.0f : vl_key_float(~top);
                }
                // second round: the candidates above wv that may still be among the Vt smallest
                for (int c0 = wave * kWave; c0 < a.m; c0 += THREADS) {
                    const int slot = c0 + lane;
                    const bool has = slot < a.m;
                    const int32_t cid = has ? li[slot] : VL_MAXINT;
                    const uint8_t f = has ? flags[slot] : 0;
                    const bool ok = (f & 2) && !(f & 16) && !(ld[slot] > tv);
                    if (has && cid != VL_MAXINT && !ok && !(f & 16)) {
                        li[slot] = VL_MAXINT;
                        ld[slot] = VL_MAXFLOAT;
                    }
                    n_exact += __popcll(__ballot(ok));
                    wave_distances_lds<CPL, LPR, U>(q_row, s.vectors, s.dim, s.nchunks, cid, ok, ld + c0, order, memo_row,
                                                    s.memo_shift);
                }
                if (s.count_evals && lane == 0 && n_exact) atomicAdd(&c->evals[stripe], (unsigned long long)n_exact);
                // A row that has to evaluate more than half of the candidates it knew by bounds exactly after all
                // (they lie within the sketch's error of the queues' last slots: real neighbour lists) gives the
                // sketch up for the rest of the call.  The first iterations fill the visit queue and keep a lot, so
                // until iteration kMemoDecide only a row that evaluates nearly all of them (7 in 8) does.
                const bool weigh = t > 2 && !resample;  // (the iteration that measures the cache uses the same two counters)
                if (weigh && lane == 0) {
                    atomicAdd(&probe_asked_s, n_real);
                    atomicAdd(&probe_hits_s, n_exact);
                }
                __syncthreads();
                if (weigh && tid == 0) {
                    const bool quit = t > kMemoDecide ? 2 * probe_hits_s > probe_asked_s : 8 * probe_hits_s > 7 * probe_asked_s;
                    if (quit) {
                        s.memo_rate[row] = memo_rate;
                        word_s = memo_rate;
                        atomicAdd(&c->sketch_rows, -1);
                    }
                }
            }
        }

        // ---- which candidates can matter at all: ann.py:75-88 ----
        // search queue: only keys below its last slot can enter.  visit queue (VL slots, Vt of them just freed): every
        // key below its last live slot, plus the Vt smallest above it.  Those are at or below the Vt-th smallest of the
        // minima of the 16-lane groups, which Vt candidates of distinct groups do not exceed.  What is picked may be a
        // superset: the merges below are exact and cut by rank.  (k == wv is the visit queue's own last slot again.)
        uint32_t rest_max = 0xFFFFFFFFu;
        if (!seen_full) {
            uint32_t mine = 0xFFFFFFFFu;
            for (int i = tid; i < a.m; i += THREADS) {
                const uint64_t k = vl_make_key(li[i], ld[i]);
                const uint32_t d = (uint32_t)(k >> 32);
                if (li[i] != VL_MAXINT && k > wv && d < mine) mine = d;
            }
            mine = row16_min_u32(mine);
            if ((lane & 15) == 0) red[tid >> 4] = mine;
            __syncthreads();
            int rank;
            const uint32_t x = rank_among<kRows16>(red, &rank);
            const uint64_t last = __ballot(lane < kRows16 && rank == a.Vt - 1);
            if (last) rest_max = (uint32_t)__builtin_amdgcn_readlane((int)x, __builtin_ctzll(last));
        }
        for (int c0 = wave * kWave; c0 < a.m; c0 += THREADS) {
            const int slot = c0 + lane;
            bool want = false;
            uint64_t k = 0;
            if (slot < a.m && li[slot] != VL_MAXINT) {
                k = vl_make_key(li[slot], ld[slot]);
                want = k < ws || (!seen_full && k != wv && (k < wv || (uint32_t)(k >> 32) <= rest_max));
            }
            const uint64_t all = __ballot(want);
            if (all == 0) continue;
            int base = 0;
            if (lane == 0) base = atomicAdd(&n_keys_s, __popcll(all));
            base = __builtin_amdgcn_readfirstlane(base);
            if (want) keys[base + __popcll(all & ((1ull << lane) - 1))] = k;
        }
        __syncthreads();
        const int n_keys = same_in_all<kShortRows>(n_keys_s);

        // ---- the survivors' places in the queues; the new ones among them ----
        const int top = 1 << (31 - __builtin_clz(max(a.L, nva)));
        auto look_up = [&](int j, uint64_t *k, int *in_q, int *in_v, bool *new_q, bool *new_v) {
            *k = j < n_keys ? keys[j] : kPadKey;
            two_lower_bounds(qa, a.L, in_q, va, nva, in_v, top, *k);
            *new_q = j < n_keys && *k < ws && qa[min(*in_q, a.L - 1)] != *k;           // not queued already
            if (*new_q)
                for (int e = 0; e < n_ex; ++e)
                    if (exl[e] == vl_key_id(*k)) *new_q = false;                       // queue.py:52-53
            *new_v = j < n_keys && !seen_full && (*in_v >= nva || va[*in_v] != *k);
        };
        auto collect = [&](bool mine, uint64_t k, uint64_t *to, int *n) {
            const uint64_t all = __ballot(mine);
            if (all == 0) return;
            int base = 0;
            if (lane == 0) base = atomicAdd(n, __popcll(all));
            base = __builtin_amdgcn_readfirstlane(base);
            if (mine) to[base + __popcll(all & ((1ull << lane) - 1))] = k;
        };
        uint64_t k0 = kPadKey;
        int in_q0 = 0, in_v0 = 0;
        bool new_q0 = false, new_v0 = false;
        for (int j0 = 0; j0 + wave * kWave < n_keys; j0 += THREADS) {
            uint64_t k;
            int in_q, in_v;
            bool new_q, new_v;
            look_up(j0 + tid, &k, &in_q, &in_v, &new_q, &new_v);
            if (j0 == 0) {
                k0 = k;
                in_q0 = in_q;
                in_v0 = in_v;
                new_q0 = new_q;
                new_v0 = new_v;
            }
            collect(new_q, k, to_search, &n_search_s);
            collect(new_v, k, to_visit, &n_fresh_s);
        }
        __syncthreads();
        const int n_search = same_in_all<kShortRows>(n_search_s), n_fresh = same_in_all<kShortRows>(n_fresh_s);

        // ---- search_queue.insert (ann.py:75-80) and visit_queue.insert (ann.py:85-88) ----
        auto put_search = [&](int r, uint64_t k) {
            if constexpr (WINDOW) {
                qa_next[r] = k;
            } else {
                qi[r] = vl_key_id(k);
                qd[r] = vl_key_dist(k);
            }
        };
        auto put_visit = [&](int r, uint64_t k) {
            if constexpr (WINDOW) {
                vq_next[r] = k;
            } else {
                vi[r] = vl_key_id(k);
                vd[r] = vl_key_dist(k);
            }
        };
        bool diff = false;
        if (n_search)
            for (int i = tid; i < a.L; i += THREADS) {
                const uint64_t k = qa[i];
                const int r = i + count_below<kAtOnce>(to_search, n_search, k);
                if (r < a.L && (WINDOW || r != i)) put_search(r, k);
            }
        if (!seen_full)
            for (int i = tid; i < nva; i += THREADS) {
                const uint64_t k = va[i];
                const int r = i + count_below<kAtOnce>(to_visit, n_fresh, k);
                if (r < a.VL && (WINDOW || r != a.Vt + i)) put_visit(r, k);
            }
        for (int j0 = 0; j0 < n_keys; j0 += THREADS) {
            if (j0 > 0) look_up(j0 + tid, &k0, &in_q0, &in_v0, &new_q0, &new_v0);
            if (new_q0) {
                const int r = in_q0 + count_below<kAtOnce>(to_search, n_search, k0);
                if (r < a.L) {
                    put_search(r, k0);
                    diff = true;  // a new id inside the first L slots: the row changed (queue.py:57-59)
                }
            }
            if (new_v0) {
                const int r = in_v0 + count_below<kAtOnce>(to_visit, n_fresh, k0);
                if (r < a.VL) put_visit(r, k0);
            }
        }
        if (!seen_full)
            for (int r = nva + n_fresh + tid; r < a.VL; r += THREADS)  // the popped slots end up here, empty
                put_visit(r, vl_make_key(VL_MAXINT, VL_MAXFLOAT));

        int *flag = &c->changed[(t / a.readahead) & 63];  // every writer stores the same 1: no atomic needed
        if (a.row_quiet) {
            // Per-query stop: a row is finished after `readahead` iterations in a row that left its first L
            // slots as they were, or when the visited list has no free column (no pop yields a real id from
            // then on); a row that is not finished at a checking iteration keeps the loop going.
            if (diff) changed_s = 1;  // every writer stores the same 1
            __syncthreads();
            if (tid == 0) {
                int quiet = changed_s ? 0 : quiet_s + 1;
                if (seen_full) quiet = a.readahead;
                quiet_s = quiet;
                if constexpr (!WINDOW) a.row_quiet[row] = quiet;
                if (checking && quiet < a.readahead &&
                    __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
                    __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        } else if (checking && __ballot(diff) && lane == 0) {
            if (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
                __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if constexpr (WINDOW) {
            // the candidates leave the set (only visited ids were in it when any of them looked for its place, so the
            // places of those stay reachable)
            for (int i = tid; i < a.m; i += THREADS)
                if (set_slot[i] != 0xffffu) set[set_slot[i]] = -1;
            cnt += same_in_all<kShortRows>(n_new_s);
            if (n_search) {
                uint64_t *const x = qa;
                qa = qa_next;
                qa_next = x;
                queue_moved = true;
            }
            uint64_t *const y = vq;
            vq = vq_next;
            vq_next = y;
            __syncthreads();
            if (a.row_quiet && quiet_s >= a.readahead) break;  // the row has stopped on its own (uniform)
        }
    }
    if constexpr (WINDOW) {
        // the row goes back to memory once
        if (queue_moved)
            for (int i = tid; i < a.L; i += THREADS) {
                qi[i] = vl_key_id(qa[i]);
                qd[i] = vl_key_dist(qa[i]);
            }
        for (int i = tid; i < a.VL; i += THREADS) {
            vi[i] = vl_key_id(vq[i]);
            vd[i] = vl_key_dist(vq[i]);
        }
        if (tid == 0) {
            if (a.row_quiet) a.row_quiet[row] = quiet_s;
            raise_running_max(first_after, cnt, bound_after);
        }
    }
}
