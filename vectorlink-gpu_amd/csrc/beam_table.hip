// The iteration of closest_vectors (ann.py:68-88) for calls that have the distances of all their queries and vectors at
// hand: what the step of beam_row.h does, without anything to evaluate.  A row is one wavefront.  Its two queues stay in
// registers, slot i in lane i mod 64 of the (i / 64)-th key; a key is read by all lanes at once, so the places of a new key
// and of the keys behind it are one comparison each per 64 slots, and LDS only carries keys to their new lanes.
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
__device__ __forceinline__ uint64_t lane_key(uint64_t k, int lane) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)k, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(k >> 32), lane);
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ int below(uint64_t mask) {  // lanes of the mask before this one
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}
// Slot `at` of a queue (the same in all lanes, and all lanes are here: what is read is chosen by every lane).
template <int N>
__device__ __forceinline__ uint64_t slot_key(const uint64_t (&k)[N], int at) {
    uint64_t x = lane_key(k[0], at & 63);
#pragma unroll
    for (int r = 1; r < N; ++r)
        if ((at >> 6) == r) x = lane_key(k[r], at & 63);
    return x;
}

template <int QR, int VR, int CR>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(CR == 8 ? 6 : 8))) void beam_table_kernel(TableStepArgs s) {
    __shared__ uint64_t moved_q[QR * 64], moved_v[VR * 64];  // keys on their way to new slots
    __shared__ uint64_t picked[64];
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
    int32_t excluded;

    // (every read that depends on nothing goes out first)
    const int unordered = *s.unordered;
    int cnt = a.seen_count[row];
    int quiet = a.row_quiet ? a.row_quiet[row] : 0;
    uint64_t qk[QR], vk[VR];
    {
        int32_t ids[QR + VR];
        float ds[QR + VR];
#pragma unroll
        for (int r = 0; r < QR + VR; ++r) {
            const int i = (r < QR ? r : r - QR) * 64 + lane;
            const bool has = i < (r < QR ? a.L : a.VL);
            ids[r] = has ? (r < QR ? qi[i] : vi[i]) : -1;
            ds[r] = has ? (r < QR ? qd[i] : vd[i]) : 0.0f;
        }
        const int32_t excluded_id = a.excl && lane < a.excl_cols ? a.excl[row * a.excl_cols + lane] : VL_MAXINT;
        excluded = excluded_id;
#pragma unroll
        for (int r = 0; r < QR; ++r) qk[r] = r * 64 + lane < a.L ? vl_make_key(ids[r], ds[r]) : kPadKey;
#pragma unroll
        for (int r = 0; r < VR; ++r) vk[r] = r * 64 + lane < a.VL ? vl_make_key(ids[QR + r], ds[QR + r]) : kPadKey;
    }
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
    if (s.enter) {
#pragma unroll
        for (int r = 0; r < VR; ++r)
            if (r * 64 + lane < a.VL && known(vl_key_id(vk[r]))) table[column.of(vl_key_id(vk[r]))] = kTableTaken;
        for (int i = lane; i < cnt; i += 64)
            if (known(srow[i])) table[column.of(srow[i])] = kTableTaken;
    }
    const uint64_t kEmpty = vl_make_key(VL_MAXINT, VL_MAXFLOAT);
    bool queue_moved = false;

    for (int w = 0; w < s.window; ++w) {
        const int t = t0 + w;
        const bool checking = (t % a.readahead) == 0;
        wave_order();  // what the last iteration wrote comes before what this one reads

        // ---- pop: queue.py:87-95; the popped ids become visited: utils.py:61-82 (there is room in these iterations) ----
        const int32_t head = lane < a.Vt ? vl_key_id(vk[0]) : VL_MAXINT;
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
        for (int r = 0; r < CR; ++r) d[r] = known(id[r]) ? table[column.of(id[r])] : kTableTaken;
        if (s.count_wanted) {
            int n = 0;
#pragma unroll
            for (int r = 0; r < CR; ++r) n += __popcll(__ballot(known(id[r])));
            if (lane == 0) atomicAdd(&c->wanted[row & (kBeamStripes - 1)], (unsigned long long)n);
        }
        auto key = [&](int r) { return ((uint64_t)(d[r] | 0x80000000u) << 32) | (uint32_t)id[r]; };  // vl_make_key of distances

        // ---- which of them can matter: keys below a queue's last slot, and the Vt smallest beyond the visit queue's (it has
        // just lost Vt).  Vt distinct distances among the lanes' smallest beyond it bound those.
        const uint64_t ws = slot_key(qk, a.L - 1), wv = slot_key(vk, a.VL - 1);
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
        bool diff = false, more = true;
        int drop = a.Vt;  // the popped heads, until they have left their slots
        for (bool first = true; more; first = false) {
            int total = 0;
#pragma unroll
            for (int r = 0; r < CR; ++r) {
                const uint64_t all = __ballot(want[r]);
                const int at = total + below(all);
                if (want[r] && at < 64) {
                    picked[at] = key(r);
                    want[r] = false;
                }
                total += __popcll(all);
            }
            more = total > 64;
            wave_order();
            const int n = min(64, total);
            const uint64_t k = lane < n ? picked[lane] : kPadKey;
            const uint64_t last_q = slot_key(qk, a.L - 1), last_v = drop > 0 ? kEmpty : slot_key(vk, a.VL - 1);
            bool in_q = lane < n && k < last_q;
            const bool in_v = lane < n && k < last_v;
            for (int e = 0; e < n_ex; ++e) in_q = in_q && vl_key_id(k) != __builtin_amdgcn_readlane(excluded, e);  // queue.py:52-53
            uint64_t to_q = __ballot(in_q), to_v = __ballot(in_v);
            const uint64_t not_popped = drop > 0 ? ~((1ull << drop) - 1) : ~0ull;
            int shift_q[QR], shift_v[VR], at_q = 0, at_v = 0;
#pragma unroll
            for (int r = 0; r < QR; ++r) shift_q[r] = 0;
#pragma unroll
            for (int r = 0; r < VR; ++r) shift_v[r] = 0;
            for (uint64_t todo = to_q | to_v; todo; todo &= todo - 1) {
                const int j = __builtin_ctzll(todo);
                const uint64_t kj = lane_key(k, j);
                const uint64_t bit = 1ull << j;
                if (__ballot(k == kj) & (bit - 1)) {  // a later copy of an id
                    to_q &= ~bit;
                    to_v &= ~bit;
                    continue;
                }
                const bool after = k > kj;
                if (to_q & bit) {
                    uint64_t same = 0;
#pragma unroll
                    for (int r = 0; r < QR; ++r) same |= __ballot(qk[r] == kj);
                    if (same) {  // queued already
                        to_q &= ~bit;
                    } else {
                        int beyond = 0;
#pragma unroll
                        for (int r = 0; r < QR; ++r) {
                            const bool g = qk[r] > kj;
                            shift_q[r] += g;
                            beyond += __popcll(__ballot(g));
                        }
                        at_q += after;
                        if (lane == j) at_q += 64 * QR - beyond;
                    }
                }
                if (!first && (to_v & bit)) {  // the copy before it may have been one of the 64 before
                    uint64_t same = 0;
#pragma unroll
                    for (int r = 0; r < VR; ++r) same |= __ballot(vk[r] == kj);
                    if (same) to_v &= ~bit;
                }
                if (to_v & bit) {
                    int beyond = 0;
#pragma unroll
                    for (int r = 0; r < VR; ++r) {
                        const bool g = vk[r] > kj;
                        shift_v[r] += g;
                        beyond += __popcll(__ballot(g) & (r == 0 ? not_popped : ~0ull));
                    }
                    at_v += after;
                    if (lane == j) at_v += 64 * VR - drop - beyond;
                }
            }
            if (to_q) {
#pragma unroll
                for (int r = 0; r < QR; ++r) {
                    const int p = r * 64 + lane + shift_q[r];
                    if (p < a.L) moved_q[p] = qk[r];
                }
                if (((to_q >> lane) & 1) && at_q < a.L) {
                    moved_q[at_q] = k;
                    diff = true;  // a new id inside the first L slots: the row changed (queue.py:57-59)
                }
                wave_order();
#pragma unroll
                for (int r = 0; r < QR; ++r)
                    if (r * 64 + lane < a.L) qk[r] = moved_q[r * 64 + lane];
                queue_moved = true;
            }
            if (to_v || drop > 0) {
                const int filled = a.VL - drop + __popcll(to_v);
#pragma unroll
                for (int r = 0; r < VR; ++r) {
                    const int i = r * 64 + lane, p = i - drop + shift_v[r];
                    if (i >= drop && i < a.VL) {
                        if (p < a.VL) moved_v[p] = vk[r];
                        else if (known(vl_key_id(vk[r]))) table[column.of(vl_key_id(vk[r]))] = (uint32_t)(vk[r] >> 32) & 0x7fffffffu;
                    }
                    if (i >= filled && i < a.VL) moved_v[i] = kEmpty;  // the popped slots end up here
                }
                if (((to_v >> lane) & 1) && at_v < a.VL) {
                    moved_v[at_v] = k;
                    table[column.of(vl_key_id(k))] = kTableTaken;
                }
                wave_order();
#pragma unroll
                for (int r = 0; r < VR; ++r)
                    if (r * 64 + lane < a.VL) vk[r] = moved_v[r * 64 + lane];
                drop = 0;
            }
            wave_order();
            if (more) {  // uniform
                const uint64_t last_q = slot_key(qk, a.L - 1), last_v = slot_key(vk, a.VL - 1);
#pragma unroll
                for (int r = 0; r < CR; ++r) {
                    const uint64_t k = key(r);
                    want[r] = want[r] && (k < last_q || k < last_v);
                }
            }
        }

        // ---- progress: ann.py:90-91, or the row's own (VL_BEAM_PER_QUERY_STOP) ----
        int *const flag = &c->changed[(t / a.readahead) & 63];  // every writer stores the same 1: no atomic needed
        const bool changed = __ballot(diff) != 0;
        bool raise = checking && changed;
        if (a.row_quiet) {
            quiet = changed ? 0 : quiet + 1;
            raise = checking && quiet < a.readahead;
        }
        if (raise && lane == 0 && __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
            __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (a.row_quiet && quiet >= a.readahead) break;
    }

    if (queue_moved) {
#pragma unroll
        for (int r = 0; r < QR; ++r)
            if (r * 64 + lane < a.L) {
                qi[r * 64 + lane] = vl_key_id(qk[r]);
                qd[r * 64 + lane] = vl_key_dist(qk[r]);
            }
    }
#pragma unroll
    for (int r = 0; r < VR; ++r)
        if (r * 64 + lane < a.VL) {
            vi[r * 64 + lane] = vl_key_id(vk[r]);
            vd[r * 64 + lane] = vl_key_dist(vk[r]);
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
