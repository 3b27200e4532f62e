// The iteration of closest_vectors (ann.py:68-88) for calls that have the distances of all their queries and vectors at
// hand: what the step of beam_row.h does, without anything to evaluate.  A row is one wavefront, its two queues are in LDS.  Up
// to 64 candidates that can matter come in at a time, a lane each: their lower bounds in the queues are searched together,
// their ranks among themselves are counted, and a queue takes them over by writing them to their slots and closing up around
// them.  (One after the other, with the queues in registers and two instructions for each 64 slots of them, a candidate took
// 560 cycles: 12 of them 6,970 of a lone wavefront's 10,350 an iteration, 60 of them 31,300 in the first ones.  256 queries at
// 4,096 x 128 564 -> 514 us, 37 at 20,011 x 50 682 -> 575, first-loop batches at 4,096 x 128 1.31 -> 1.17 ms, 6,007 x 384 2.85 ->
// 2.52, 20,011 x 768 12.5 -> 11.8, where a launch of five iterations moves 0.53 GB past L2 in 118 us, 4.5 TB/s, most of it the
// table's cache lines.)
//
// An entry of the row's table is taken while its id sits in the visit queue and from the moment it was visited.  Such a
// candidate can change neither queue (beam_row.h says why for visited ones; one in the visit queue was offered to the search
// queue with this distance when it came), so a candidate costs one look at the table and most are through after it.  What
// falls off the end of the visit queue becomes an ordinary entry again: it may come back when the queue has room.
//
// The accesses of one wavefront to its row of the table reach its cache in the order in which it makes them.
#include "beam_table.h"
#include "pair_table.h"

namespace {

constexpr uint32_t kTableTaken = 0xFFFFFFFFu;

__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ int below(uint64_t mask) {  // lanes of the mask before this one
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}
// How many of a sorted queue's 64 R slots hold a smaller key (slots past its end hold kPadKey; not all of them do).  Two trips
// to LDS take a power of two of the slots away where a binary search takes one: quarters of a quarter of a set of 64.
template <int R>
__device__ __forceinline__ int keys_below(const uint64_t *q, uint64_t k) {
    int at = 0;
#pragma unroll
    for (int r = 1; r < R; ++r) at += q[64 * r - 1] < k ? 64 : 0;
#pragma unroll
    for (int step = 16; step > 0; step >>= 2) {
        const uint64_t x = q[at + step - 1], y = q[at + 2 * step - 1], z = q[at + 3 * step - 1];
        at += (x < k ? step : 0) + (y < k ? step : 0) + (z < k ? step : 0);
    }
    return at;
}
// How many of n keys in LDS (n the same in all lanes) are smaller; four reads are on their way at a time.
__device__ __forceinline__ int count_less(const uint64_t *keys, int n, uint64_t k) {
    int c = 0;
    for (int i = 0; i < n; i += 4) {
        uint64_t x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = keys[i + j];  // (kPadKey past the last)
#pragma unroll
        for (int j = 0; j < 4; ++j) c += x[j] < k;
    }
    return c;
}

template <int QR, int VR, int CR>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(CR == 8 ? 6 : 7))) void beam_table_kernel(TableStepArgs s) {
    __shared__ uint64_t queue[QR * 64], visit[VR * 64 + kTableMaxVisit];  // kPadKey past their ends
    __shared__ uint64_t placed_q[QR * 64], placed_v[VR * 64];  // the new keys in their slots, 0 elsewhere
    uint64_t *const picked_q = placed_q, *const picked_v = placed_v;  // before that: the new keys as they come
    __shared__ uint8_t owner[(QR > VR ? QR : VR) * 64];               // whose key a slot took
    const MergeArgs &a = s.m;
    BeamCtrl *const c = a.ctrl;
    const int t0 = a.iter;
    const int lane = threadIdx.x;
    const int64_t row = blockIdx.x;
    const bool writer = row == 0 && lane == 0;
    int32_t *const vi = a.v_ids + row * a.VL;
    float *const vd = a.v_d + row * a.VL;
    int32_t *const qi = a.q_ids + row * a.cap;
    float *const qd = a.q_d + row * a.cap;
    int32_t *const srow = a.seen + row * a.E;
    uint32_t *const table = s.table + row * s.columns;
    const int seen_bound = min(a.E, a.Vt * (t0 - 1));

    // (every read that depends on nothing goes out first)
    const int unordered = *s.unordered;
    int cnt = a.seen_count[row];
    int quiet = a.row_quiet ? a.row_quiet[row] : 0;
    int32_t ids[QR + VR];
    float ds[QR + VR];
#pragma unroll
    for (int r = 0; r < QR + VR; ++r) {
        const int i = (r < QR ? r : r - QR) * 64 + lane;
        const bool has = i < (r < QR ? a.L : a.VL);
        ids[r] = has ? (r < QR ? qi[i] : vi[i]) : VL_MAXINT;
        ds[r] = has ? (r < QR ? qd[i] : vd[i]) : VL_MAXFLOAT;
    }
    const int32_t excluded = a.excl && lane < a.excl_cols ? a.excl[row * a.excl_cols + lane] : VL_MAXINT;
    const int gate = unordered ? 0 : beam_gate(c, t0, a.readahead, a.E, writer, s.report, false);
    if (unordered) {  // (nothing of this launch happens; the loop goes on without a table from iteration t0)
        if (writer) {
            if (c->refused_at == 0) c->refused_at = t0;
            if (s.report && t0 > 1) beam_report(c, t0 - 1, a.readahead, s.report);
        }
        return;
    }
    if (gate == 2) return;
    cnt = __builtin_amdgcn_readfirstlane(cnt);
    quiet = __builtin_amdgcn_readfirstlane(quiet);
    if (!beam_row_state_ok(c, cnt, seen_bound, lane == 0)) return;
    const uint64_t ends = __ballot(excluded == VL_MAXINT);  // a row's exclusions end at its first empty one
    const int n_ex = ends ? __builtin_ctzll(ends) : 64;
    int *const first_after = &c->first[(t0 + s.window) % 3];
    const int bound_after = min(a.E, a.Vt * (t0 + s.window - 1));
    if (a.row_quiet && quiet >= a.readahead) {
        if (s.raise_fill && lane == 0) raise_running_max(first_after, cnt, bound_after);
        return;
    }
    auto known = [&](int32_t id) { return id >= 0 && (int64_t)id < s.n_vectors; };  // (VL_MAXINT is beyond every table)
    const PairColumns column(s.n_vectors);
    auto entry = [&](int32_t id) -> uint32_t & { return table[column.of((uint32_t)id)]; };
#pragma unroll
    for (int r = 0; r < QR + VR; ++r) {
        const int i = (r < QR ? r : r - QR) * 64 + lane;
        (r < QR ? queue : visit)[i] = i < (r < QR ? a.L : a.VL) ? vl_make_key(ids[r], ds[r]) : kPadKey;
    }
    if (lane < kTableMaxVisit) visit[VR * 64 + lane] = kPadKey;
    if (s.enter) {
#pragma unroll
        for (int r = QR; r < QR + VR; ++r)
            if (known(ids[r])) entry(ids[r]) = kTableTaken;
        for (int i = lane; i < cnt; i += 64)
            if (known(srow[i])) entry(srow[i]) = kTableTaken;
    }
    const uint64_t kEmpty = vl_make_key(VL_MAXINT, VL_MAXFLOAT);
    bool queue_moved = false;

    for (int w = 0; w < s.window; ++w) {
        const int t = t0 + w;
        const bool checking = (t % a.readahead) == 0;
        wave_order();  // what the last iteration wrote comes before what this one reads

        // ---- pop: queue.py:87-95; the popped ids become visited: utils.py:61-82 (there is room in these iterations) ----
        const int32_t head = lane < a.Vt ? vl_key_id(visit[lane]) : VL_MAXINT;
        const uint64_t heads = __ballot(head != VL_MAXINT);
        if (head != VL_MAXINT) srow[cnt + below(heads)] = head;
        cnt += __popcll(heads);

        // ---- the candidates and their distances: ann.py:69-73 ----
        int32_t id[CR];
#pragma unroll
        for (int r = 0; r < CR; ++r) {
            const int slot = r * 64 + lane;
            id[r] = VL_MAXINT;
            if (r * 64 < a.m) {  // uniform
                const int of = s.width == 1 ? slot : (int)__umulhi((uint32_t)slot, s.width_magic);
                const int32_t node = __shfl(head, of & 63);
                if (slot < a.m && known(node)) id[r] = s.beams[(int64_t)node * s.width + (slot - of * s.width)];
            }
        }
        uint32_t d[CR];
#pragma unroll
        for (int r = 0; r < CR; ++r) d[r] = known(id[r]) ? entry(id[r]) : kTableTaken;
        if (s.count_wanted) {
            int n = 0;
#pragma unroll
            for (int r = 0; r < CR; ++r) n += __popcll(__ballot(known(id[r])));
            if (lane == 0) atomicAdd(&c->wanted[row & (kBeamStripes - 1)], (unsigned long long)n);
        }
        auto key = [&](int r) { return ((uint64_t)(d[r] | 0x80000000u) << 32) | (uint32_t)id[r]; };  // vl_make_key of distances

        // ---- which of them can matter: keys below a queue's last slot, and the Vt smallest beyond the visit queue's (it has
        // just lost Vt).  Vt distinct distances among the lanes' smallest beyond it bound those.
        const uint64_t ws = queue[a.L - 1], wv = visit[a.VL - 1];
        uint32_t least = kTableTaken, bound = kTableTaken - 1;
#pragma unroll
        for (int r = 0; r < CR; ++r) {
            const uint64_t k = key(r);
            const uint32_t hi = (uint32_t)(k >> 32);
            least = k > wv && hi < least ? hi : least;
        }
        for (int i = 0; i < a.Vt; ++i) {
            const uint32_t x = wave_min_u32(least);
            bound = x == kTableTaken ? kTableTaken - 1 : x;
            if (x == kTableTaken) break;  // uniform
            least = least == x ? kTableTaken : least;
        }
        bool want[CR];
#pragma unroll
        for (int r = 0; r < CR; ++r) {
            const uint64_t k = key(r);
            want[r] = k < ws || k < wv || (uint32_t)(k >> 32) <= bound;
        }

        // ---- search_queue.insert (ann.py:75-80) and visit_queue.insert (ann.py:85-88), up to 64 candidates at a time; what
        // the ones before have put out of reach is left alone
        bool changed = false, more = true;
        int drop = a.Vt;  // the popped heads, until they have left their slots
        for (bool first = true; more; first = false) {
            int total = 0;
#pragma unroll
            for (int r = 0; r < CR; ++r) {
                const uint64_t all = __ballot(want[r]);
                const int at = total + below(all);
                if (want[r] && at < 64) {
                    picked_v[at] = key(r);
                    want[r] = false;
                }
                total += __popcll(all);
            }
            more = total > 64;
            wave_order();
            const int n = min(64, total);
            const uint64_t k = lane < n ? picked_v[lane] : kPadKey;
            const int below_q = keys_below<QR>(queue, k), below_v = keys_below<VR>(visit + drop, k);
            bool in_q = k < queue[a.L - 1] && queue[min(below_q, a.L - 1)] != k;             // not queued already
            bool in_v = lane < n && (drop > 0 || k < visit[a.VL - 1]);
            if (!first) in_v = in_v && visit[min(below_v, a.VL - 1)] != k;  // (its other copy may have been one of the 64 before)
            for (int e = 0; e < n_ex; ++e) in_q = in_q && vl_key_id(k) != __builtin_amdgcn_readlane(excluded, e);  // queue.py:52-53
            // To their slots: smaller new keys come before.  Copies of an id share a slot, which shows in the number of
            // slots taken; one of them stays, and the places are found again.
            bool place_q, place_v;
            uint64_t new_q, new_v, now_q[QR], now_v[VR];
            for (;;) {
                const uint64_t to_q = __ballot(in_q), to_v = __ballot(in_v);
                if (lane < ((n + 3) & ~3)) {
                    picked_q[lane] = in_q ? k : kPadKey;
                    picked_v[lane] = in_v ? k : kPadKey;
                }
                wave_order();
                const int at_q = below_q + (to_q ? count_less(picked_q, n, k) : 0);
                const int at_v = below_v + (to_v ? count_less(picked_v, n, k) : 0);
                place_q = in_q && at_q < a.L;
                place_v = in_v && at_v < a.VL;
                new_q = __ballot(place_q);
                new_v = __ballot(place_v);
                wave_order();
                if (new_q) {
#pragma unroll
                    for (int r = 0; r < QR; ++r) placed_q[r * 64 + lane] = 0;
                }
                if (new_v) {
#pragma unroll
                    for (int r = 0; r < VR; ++r) placed_v[r * 64 + lane] = 0;
                }
                wave_order();
                if (place_q) placed_q[at_q] = k;
                if (place_v) placed_v[at_v] = k;
                wave_order();
                int taken = 0;
#pragma unroll
                for (int r = 0; r < QR; ++r) {
                    now_q[r] = new_q ? placed_q[r * 64 + lane] : 0;
                    taken += __popcll(__ballot(now_q[r] != 0));
                }
#pragma unroll
                for (int r = 0; r < VR; ++r) {
                    now_v[r] = new_v ? placed_v[r * 64 + lane] : 0;
                    taken += __popcll(__ballot(now_v[r] != 0));
                }
                if (taken == __popcll(new_q) + __popcll(new_v)) break;
                if (place_v) owner[at_v] = (uint8_t)lane;
                wave_order();
                const bool copy_v = place_v && owner[at_v] != lane;
                wave_order();
                if (place_q) owner[at_q] = (uint8_t)lane;
                wave_order();
                if (copy_v || (place_q && !place_v && owner[at_q] != lane)) in_q = in_v = false;
                wave_order();
            }
            changed = changed || new_q != 0;  // a new id inside the first L slots: the row changed (queue.py:57-59)
            if (place_v) entry(vl_key_id(k)) = kTableTaken;
            // the keys that were there close up around them
            if (new_q) {
                int taken = 0;
#pragma unroll
                for (int r = 0; r < QR; ++r) {
                    const uint64_t all = __ballot(now_q[r] != 0), y = queue[r * 64 + lane - taken - below(all)];
                    now_q[r] = now_q[r] ? now_q[r] : y;
                    taken += __popcll(all);
                }
            }
            if (new_v || drop > 0) {
                int taken = 0;
#pragma unroll
                for (int r = 0; r < VR; ++r) {
                    const uint64_t all = __ballot(now_v[r] != 0);
                    const int from = r * 64 + lane - taken - below(all) + drop;
                    const uint64_t y = visit[min(from, a.VL - 1)];
                    now_v[r] = now_v[r] ? now_v[r] : from < a.VL ? y : kEmpty;  // the popped slots end up at the end, empty
                    taken += __popcll(all);
                }
                if (lane < taken - drop) {  // these fall off the end
                    const uint64_t x = visit[a.VL - 1 - lane];
                    if (known(vl_key_id(x))) entry(vl_key_id(x)) = (uint32_t)(x >> 32) & 0x7fffffffu;
                }
            }
            wave_order();
            if (new_q) {
#pragma unroll
                for (int r = 0; r < QR; ++r)
                    if (r * 64 + lane < a.L) queue[r * 64 + lane] = now_q[r];
                queue_moved = true;
            }
            if (new_v || drop > 0) {
#pragma unroll
                for (int r = 0; r < VR; ++r)
                    if (r * 64 + lane < a.VL) visit[r * 64 + lane] = now_v[r];
                drop = 0;
            }
            wave_order();
            if (more) {  // uniform
                const uint64_t last_q = queue[a.L - 1], last_v = visit[a.VL - 1];
#pragma unroll
                for (int r = 0; r < CR; ++r) {
                    const uint64_t k = key(r);
                    want[r] = want[r] && (k < last_q || k < last_v);
                }
            }
        }

        // ---- progress: ann.py:90-91, or the row's own (VL_BEAM_PER_QUERY_STOP) ----
        int *const flag = &c->changed[(t / a.readahead) & 63];  // every writer stores the same 1: no atomic needed
        bool raise = checking && changed;
        if (a.row_quiet) {
            quiet = changed ? 0 : quiet + 1;
            raise = checking && quiet < a.readahead;
        }
        if (raise && lane == 0 && __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
            __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (a.row_quiet && quiet >= a.readahead) break;
    }

    if (queue_moved)
        for (int i = lane; i < a.L; i += 64) {
            qi[i] = vl_key_id(queue[i]);
            qd[i] = vl_key_dist(queue[i]);
        }
    for (int i = lane; i < a.VL; i += 64) {
        vi[i] = vl_key_id(visit[i]);
        vd[i] = vl_key_dist(visit[i]);
    }
    if (lane == 0) {
        a.seen_count[row] = cnt;
        if (a.row_quiet) a.row_quiet[row] = quiet;
        if (s.raise_fill) raise_running_max(first_after, cnt, bound_after);
    }
}

template <int QR, int VR>
void launch_by_candidates(const TableStepArgs &s, hipStream_t st) {
    const dim3 grid((unsigned)s.m.n_rows), block(64);
    if (s.m.m <= 128) hipLaunchKernelGGL((beam_table_kernel<QR, VR, 2>), grid, block, 0, st, s);
    else if (s.m.m <= 256) hipLaunchKernelGGL((beam_table_kernel<QR, VR, 4>), grid, block, 0, st, s);
    else hipLaunchKernelGGL((beam_table_kernel<QR, VR, 8>), grid, block, 0, st, s);
}
template <int QR>
void launch_by_visit(const TableStepArgs &s, hipStream_t st) {
    if (s.m.VL <= 128) launch_by_candidates<QR, 2>(s, st);
    else launch_by_candidates<QR, 3>(s, st);
}

}  // namespace

int vl_launch_table_step(const TableStepArgs &s, hipStream_t st) {
    if (s.m.L <= 64) launch_by_visit<1>(s, st);
    else if (s.m.L <= 128) launch_by_visit<2>(s, st);
    else launch_by_visit<3>(s, st);
    VL_LAUNCH_CHECK("beam_table_kernel");
    return VL_OK;
}
