// Exact k nearest neighbours of many queries for gfx950: a bfloat16 pass over all pairs finds the few vectors that can be
// among the k best of a query, and only those are evaluated in float32.
//
// The float32 tiles of knn.hip are bound by the float32 matrix rate (157 TFLOP/s; 123 reached).  bfloat16 products run
// sixteen times as fast, and all the pass has to decide is which vectors cannot matter.  With q^, v^ the rows rounded to
// bfloat16,
//   | <q, v> - <q^, v^> |  <=  ||q - q^|| ||v||  +  ||q^|| ||v - v^||          (Cauchy-Schwarz)
// and both roundings are known exactly: ||q - q^|| per query, the largest ||v|| and ||v - v^|| per piece of the table.
// With the float32 roundings of either sum (at most dim * 2^-24 of ||q|| ||v|| each; 2^-22 is used for both together) that
// is a bound E on how far a value of the pass is from the value the float32 tiles would form.  A query's k-th best value
// T over any subset bounds its k-th best over all from below, so whatever the pass gives less than T - 2E is out.
//   prepare   rows to bfloat16, their norms and roundings
//   sample    the pass over 1/16 of the table: the maximum of each of a few hundred groups per query; the k-th largest
//             of those is T (k different vectors are at least as good)
//   filter    the pass over all: ids of the values that are not out, per query
//   finish    their float32 dot products - one fused multiply-add after the other in the order in which the float32 tiles'
//             matrix instructions take the elements, which gives the tiles' bits - and the k best of them
// A query with more candidates than its buffer holds (thousands of rows within the rounding of each other), or than the
// tiles are worth (expected_limit), is left to the float32 tiles, which take all such queries of a call together; most are
// known from the sample and are not looked for in the pass.  For squared L2 the values are <q, v> - |v|^2 / 2: three more
// columns hold -|v|^2 / 2 as a sum of three bfloat16 numbers (24 bits), and ones on the query side.
//
// The pass: 256 vectors x 256 queries per workgroup of eight wavefronts (128 x 64 each, 128 accumulator registers), 64
// columns per stage through two LDS buffers per operand (128 KB), v_mfma_f32_32x32x16_bf16.  A wavefront reads 6 KB of
// LDS per 8 products of 32 cycles; with 64 x 64 per wavefront LDS (128 bytes per cycle) would be the bound.
// Measured, 10,000 queries, k = 10 (k = 4 and 16 below): 1,000,000 x 768 17.5 ms of which the pass 15.0 = 1,026 TFLOP/s
// (a library product of 16,384^3 reaches 1,345 on the same card), 124.5 ms with the float32 tiles; 32,768 x 64 0.30 ms (0.61),
// 32,768 x 128 0.44 ms (1.34), 1,000 queries at 32,768 x 1,536 0.33 ms (0.90).  What is left of the short ones is storing the
// candidates.
#include "knn_device.h"
#include "knn_filter.h"
#include "near_products.h"

#include <type_traits>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

constexpr int TR = 256;           // rows of either operand per workgroup
constexpr int kThreads = 512;
constexpr int RB = 4, CB = 2;     // 32-row and 32-column blocks of a wavefront
constexpr int kGroupsPerStrip = 2 * 2 * RB;  // maxima that a strip's workgroup leaves per query
constexpr int kFound = 2048;      // candidates per query
constexpr int kMaxGroups = 512;
constexpr int kStripes = 64, kStripeWords = 32;  // partial maxima of a piece of the table, a cache line each (in the sample's: a third word, bound_kernel)
constexpr float kMostExpected = 1.25f * kFound;  // expected candidates with which a query is still looked for: the sample is off by a tenth
// Batches of so few queries leave compute units idle: 512 threads per query evaluate its candidates instead of 128.
constexpr int64_t kFinishWide = 512;

struct RowStat {
    float resid, norm;  // not below ||x - x^||_2 and ||x||_2
};
// What the sample tells of a query.
struct alignas(16) Sampled {
    float value;       // the k-th best float32 value is not below this
    float expected;    // how many vectors the pass will not rule out
    float error;       // value_error with the sample's rows
};

__device__ __forceinline__ float up(float x) { return x * 1.00001f; }  // norms are sums of dim rounded terms: never below

// The sample takes one row of each of n_sample equal stretches of the table, at a place of its own in each, and deals
// neighbours to groups far apart: a table whose rows come in the order of their clusters, or in turn from each, is sampled
// like one in random order.  (Whole tiles at equal distances met 1 in 16 of the clusters of a table in their order, and the
// bounds from those that were met let thousands of candidates through.)
struct SampleRows {
    int64_t n_sample, n_table;
    int64_t stride;  // has no common divisor with n_sample
    __device__ __forceinline__ int64_t source(int64_t i) const {
        const int64_t first = i * n_table / n_sample, room = (i + 1) * n_table / n_sample - first;
        uint32_t h = (uint32_t)i * 2654435761u;  // (the finaliser of MurmurHash3)
        h = (h ^ (h >> 16)) * 0x85ebca6bu;
        h = (h ^ (h >> 13)) * 0xc2b2ae35u;
        return first + (int64_t)__umulhi(h ^ (h >> 16), (uint32_t)room);
    }
    __device__ __forceinline__ int64_t place(int64_t i) const { return i * stride % n_sample; }
};

// Rows of the input (all n, or a sample of n) rounded to bfloat16 and padded with zeros to kp columns.  extra: 0, 1 = a query row for L2 (three ones behind the columns), 2 = a vector for L2 (-|v|^2 / 2 there).  One wavefront per row.  vmax: the largest resid and norm as float bits (all values are >= 0; what is not
// finite counts as infinity), over kStripes stripes that table_stat puts together - with one pair of words for all, the
// 32,768 atomic operations of a large table queued up for 280 us.
template <bool SAMPLE>
__global__ __launch_bounds__(256) void prepare_kernel(const float *__restrict__ rows, int64_t n, int dim, int kp,
                                                      SampleRows sample, int extra, __bf16 *__restrict__ out,
                                                      float *__restrict__ norm2,
                                                      RowStat *__restrict__ stat, uint32_t *__restrict__ vmax) {
    const int lane = threadIdx.x & (kWave - 1);
    float top_resid = 0.0f, top_norm = 0.0f;
    for (int64_t i = (int64_t)blockIdx.x * 4 + threadIdx.x / kWave; i < n; i += (int64_t)gridDim.x * 4) {
        const int64_t row = SAMPLE ? sample.source(i) : i, j = SAMPLE ? sample.place(i) : i;
        const float4 *src = reinterpret_cast<const float4 *>(rows + row * dim);
        bf16x4 *dst = reinterpret_cast<bf16x4 *>(out + j * kp);
        float s = 0.0f, e2 = 0.0f;
        for (int c = lane; c < kp / 4; c += kWave) {
            bf16x4 h = {0, 0, 0, 0};
            if (c < dim / 4) {
                const float4 x = src[c];
                // (the order of row_norms_kernel)
                s = fmaf(x.x, x.x, s);
                s = fmaf(x.y, x.y, s);
                s = fmaf(x.z, x.z, s);
                s = fmaf(x.w, x.w, s);
                h = bf16x4{(__bf16)x.x, (__bf16)x.y, (__bf16)x.z, (__bf16)x.w};
                const float a = x.x - (float)h[0], b = x.y - (float)h[1], d = x.z - (float)h[2], e = x.w - (float)h[3];
                e2 = fmaf(a, a, e2);
                e2 = fmaf(b, b, e2);
                e2 = fmaf(d, d, e2);
                e2 = fmaf(e, e, e2);
            }
            if (extra == 0 || c != dim / 4) dst[c] = h;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            s += __shfl_xor(s, o);
            e2 += __shfl_xor(e2, o);
        }
        if (lane == 0 && norm2) norm2[j] = s;
        if (lane == 0 && extra) {
            bf16x4 h = {1.0f, 1.0f, 1.0f, 0.0f};
            if (extra == 2) {
                float left = -0.5f * s;
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    h[c] = (__bf16)left;
                    left -= (float)h[c];
                }
            }
            dst[dim / 4] = h;
        }
        float resid = up(sqrtf(e2)), norm = up(sqrtf(s));
        if (!(resid < 1e18f)) resid = __builtin_inff();  // also NaN
        if (!(norm < 1e18f)) norm = __builtin_inff();
        if (lane == 0 && stat) stat[j] = RowStat{resid, norm};
        top_resid = fmaxf(top_resid, resid);
        top_norm = fmaxf(top_norm, norm);
    }
    if (!vmax) return;
    __shared__ float part[4][2];
    if (lane == 0) {
        part[threadIdx.x / kWave][0] = top_resid;
        part[threadIdx.x / kWave][1] = top_norm;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        float top = part[0][threadIdx.x];
        for (int w = 1; w < 4; ++w) top = fmaxf(top, part[w][threadIdx.x]);
        atomicMax(vmax + (blockIdx.x & (kStripes - 1)) * kStripeWords + threadIdx.x, __builtin_bit_cast(uint32_t, top));
    }
}

// The largest resid and norm of a piece of the table, in every lane.
__device__ __forceinline__ RowStat table_stat(const uint32_t *__restrict__ vmax) {
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t *mine = vmax + lane * kStripeWords;
    // (the smallest of the inverted words is the largest word)
    return RowStat{__builtin_bit_cast(float, ~wave_min_u32(~mine[0])), __builtin_bit_cast(float, ~wave_min_u32(~mine[1]))};
}

// How far a value of the pass may be from the float32 tiles' value, plus what makes two float32 distances of different
// values equal (the rounding of 1 - s, or of the sums of an L2 distance).
__device__ __forceinline__ float value_error(RowStat q, RowStat v, int dim, bool l2) {
    const float v_resid = v.resid, v_norm = v.norm;
    const float both = (q.norm + q.resid) * (v_norm + v_resid);
    const float sums = l2 ? both + v_norm * v_norm : both;
    const float ties = l2 ? 2e-6f * (q.norm * q.norm + v_norm * v_norm) : 4e-7f;
    return up(q.resid * v_norm + (q.norm + q.resid) * v_resid) + (float)dim * 2.4e-7f * sums + ties;
}

// The expected number of candidates up to which the pass looks for a query's.  `most` candidates cost what the tiles do for
// one query of a full batch, `above` of the n queries expect more.  The tiles take as long for one query as for a few hundred, so a small
// batch is left to them as a whole, if most of its queries expect too many, or not at all; in a large one the queries
// far above, or if they are many all that are above, are left.  (32,768 x 768 in clusters of 977, k = 1, us with the tiles / the
// filter that left every query above / this: 300 queries 235 / 484 / 306, 1,000 456 / 610 / 492, 4,000 1,672 / 1,952 / 1,730.)
__device__ __forceinline__ float expected_limit(const uint32_t *__restrict__ sample_vmax, int64_t n, float most) {
    int above = (int)sample_vmax[(threadIdx.x & (kWave - 1)) * kStripeWords + 2];
    above += __builtin_amdgcn_update_dpp(0, above, 0x128, 0xf, 0xf, false);  // row_ror:8
    above += __builtin_amdgcn_update_dpp(0, above, 0x124, 0xf, 0xf, false);  // row_ror:4
    above += __builtin_amdgcn_update_dpp(0, above, 0x122, 0xf, 0xf, false);  // row_ror:2
    above += __builtin_amdgcn_update_dpp(0, above, 0x121, 0xf, 0xf, false);  // row_ror:1
    above = __builtin_amdgcn_readlane(above, 0) + __builtin_amdgcn_readlane(above, 16) + __builtin_amdgcn_readlane(above, 32) +
            __builtin_amdgcn_readlane(above, 48);
    if (n <= kFinishWide) return 2 * above > n ? -1.0f : kMostExpected;
    return 2 * above >= n ? most : fminf(2.0f * most, kMostExpected);
}

// Staging of 256-row operands by eight wavefronts: wavefront w brings rows 32 w ... 32 w + 31, eight per instruction.
__device__ __forceinline__ void stage256(const float *const (&p)[4], int kt, float *tile, int wave) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
        __builtin_amdgcn_global_load_lds((glb_void *)(p[i] + kt), (lds_void *)(tile + 8 * (4 * wave + i) * KT), 16, 0, 0);
}

// What a pass leaves of its values: the sample's groups' maxima in gmax, the filter's candidates in found, or all of them rounded to
// 16 bits (kAllValues: query by query, id0 of them each and as many vectors, whole tiles; out).
enum PassKind { kSampleMaxima, kCandidates, kAllValues };
// Rows are bfloat16 of kp columns, addressed as floats (two columns each); a stage is KT floats = 64 columns.
template <PassKind KIND>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void pass_kernel(const float *__restrict__ q16, int64_t n_queries, const float *__restrict__ v16, int64_t n_vectors,
                 int kp2, int64_t strip_len, int n_strips, int n_qblocks, int q_group, float *__restrict__ gmax,
                 const Sampled *__restrict__ bound, const RowStat *__restrict__ qstat, const uint32_t *__restrict__ vmax,
                 const uint32_t *__restrict__ sample_vmax, float most, int dim, int l2,
                 int64_t id0, int32_t *__restrict__ count, uint64_t *__restrict__ found, uint16_t *__restrict__ out) {
    constexpr bool EMIT = KIND == kCandidates;
    extern __shared__ __align__(16) float smem[];
    constexpr int T = TR * KT;  // floats of a staged operand
    float *const sV0 = smem, *const sV1 = smem + T, *const sQ0 = smem + 2 * T, *const sQ1 = smem + 3 * T;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave >> 2, wc = wave & 3;  // 2 x 4 wavefronts
    const int half = lane >> 5, l32 = lane & 31;
    // work items in the order of knn_tile_kernel: q_group query blocks go through the strips together, an eighth of the
    // order per XCD
    int q_block, strip;
    {
        const int64_t total = (int64_t)n_qblocks * n_strips;
        const int64_t per_xcd = (total + 7) >> 3;
        const int64_t j = blockIdx.x >> 3;
        const int64_t t = (int64_t)(blockIdx.x & 7) * per_xcd + j;
        if (j >= per_xcd || t >= total) return;
        const int64_t full = (int64_t)(n_qblocks / q_group) * q_group * n_strips;
        if (t < full) {
            const int64_t per_group = (int64_t)q_group * n_strips;
            const int64_t g = t / per_group, w = t - g * per_group;
            strip = (int)(w / q_group);
            q_block = (int)(g * q_group + (w - (int64_t)strip * q_group));
        } else {
            const int rest = n_qblocks % q_group;
            const int64_t w = t - full;
            strip = (int)(w / rest);
            q_block = (n_qblocks / q_group) * q_group + (int)(w - (int64_t)strip * rest);
        }
    }
    const int64_t q0 = (int64_t)q_block * TR;
    const int64_t v_begin = (int64_t)strip * strip_len;
    const int64_t v_end = min(n_vectors, v_begin + strip_len);

    float thr[CB], top[CB][RB];
    RowStat table = {0.0f, 0.0f}, q_stat[CB];
    float limit = 0.0f;
    Sampled sampled[CB];
    if constexpr (EMIT) {
        // (read without conditions, so that one round trip to memory brings all of it)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            const int64_t q = min(q0 + 64 * wc + 32 * cb + l32, n_queries - 1);
            sampled[cb] = bound[q];
            q_stat[cb] = qstat[q];
        }
        table = table_stat(vmax);
        limit = expected_limit(sample_vmax, n_queries, most);
    }
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        if constexpr (EMIT) {
            const int64_t q = q0 + 64 * wc + 32 * cb + l32;
            thr[cb] = __builtin_inff();
            if (q < n_queries) {
                const float error = value_error(q_stat[cb], table, dim, l2 != 0);
                thr[cb] = sampled[cb].value - error;
                // Too many expected, no bound (a row that is not finite), or one that lets everything through because a row is
                // far longer than those of the sample: the query is left to the tiles.  So a threshold is above -infinity,
                // which is what rows past the strip's end hold.
                if (!(sampled[cb].expected <= limit) || !(thr[cb] > (l2 ? -__builtin_inff() : -0.999f)) || error > 16.0f * sampled[cb].error) {
                    thr[cb] = __builtin_inff();
                    if (strip == 0 && wr == 0 && half == 0) atomicAdd(&count[q], kFound + 1);
                }
            }
        }
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) top[cb][rb] = -__builtin_inff();
    }
    if constexpr (EMIT) {
        // a workgroup none of whose queries is looked for ends here (the words are in a buffer that the first stage leaves alone)
        int *const looked_for = reinterpret_cast<int *>(sQ1);
        const bool mine = __builtin_amdgcn_ballot_w64(thr[0] < __builtin_inff() || thr[1] < __builtin_inff()) != 0;
        if (lane == 0) looked_for[wave] = mine;
        __syncthreads();
        int any = 0;
#pragma unroll
        for (int w = 0; w < kThreads / kWave; ++w) any |= looked_for[w];
        if (!any) return;
    }
    int a_off[RB], b_off[CB];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        const int r = 128 * wr + 32 * i + l32;
        a_off[i] = r * (KT * 4) | ((half ^ swz(r)) << 4);
    }
#pragma unroll
    for (int i = 0; i < CB; ++i) {
        const int r = 64 * wc + 32 * i + l32;
        b_off[i] = r * (KT * 4) | ((half ^ swz(r)) << 4);
    }
    const float *qp[4], *vp[4];
    duty_pointers(q16, q0, n_queries - 1, kp2, wave, lane, qp);
    if (v_begin < v_end) {
        duty_pointers(v16, v_begin, v_end - 1, kp2, wave, lane, vp);
        stage256(vp, 0, sV0, wave);
        stage256(qp, 0, sQ0, wave);
    }

    floatx16 acc[RB][CB];
    // one stage: wait for its operands, start the next stage's loads into the other buffers, multiply
    auto stage = [&](auto which, int64_t vt, int kt) __attribute__((always_inline)) {
        constexpr int B = decltype(which)::value;
        float *const v_cur = B ? sV1 : sV0, *const q_cur = B ? sQ1 : sQ0;
        float *const v_nxt = B ? sV0 : sV1, *const q_nxt = B ? sQ0 : sQ1;
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
        __syncthreads();
        int nkt = kt + KT;
        bool has_next = true;
        if (nkt >= kp2) {
            nkt = 0;
            has_next = vt + TR < v_end;
            if (has_next) duty_pointers(v16, vt + TR, v_end - 1, kp2, wave, lane, vp);
        }
        if (has_next) {
            stage256(vp, nkt, v_nxt, wave);
            stage256(qp, nkt, q_nxt, wave);
        }
        const char *tv = reinterpret_cast<const char *>(v_cur);
        const char *tq = reinterpret_cast<const char *>(q_cur);
        bf16x8 a0[RB], b0[CB], a1[RB], b1[CB];
        auto read = [&](bf16x8 (&a)[RB], bf16x8 (&b)[CB], int g) {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) a[rb] = *reinterpret_cast<const bf16x8 *>(tv + (a_off[rb] ^ (g << 5)));
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) b[cb] = *reinterpret_cast<const bf16x8 *>(tq + (b_off[cb] ^ (g << 5)));
            __builtin_amdgcn_sched_barrier(0);  // ahead of the products below
        };
        auto multiply = [&](const bf16x8 (&a)[RB], const bf16x8 (&b)[CB]) {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int cb = 0; cb < CB; ++cb)
                    acc[rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[rb], b[cb], acc[rb][cb], 0, 0, 0);
        };
        // operands of the next step are read while the products of this one are formed
        static_assert(KT / 8 == 4, "four steps per stage");
        read(a0, b0, 0);
        read(a1, b1, 1);
        multiply(a0, b0);
        read(a0, b0, 2);
        multiply(a1, b1);
        read(a1, b1, 3);
        multiply(a0, b0);
        multiply(a1, b1);
    };
    // accumulator register r of block rb: vector row 128 wr + 32 rb + 8 (r / 4) + 4 half + r % 4 of the tile, query l32
    auto fold = [&](int64_t vt) __attribute__((always_inline)) {
        const int64_t v_lane = vt + 128 * wr + 4 * half;
        if constexpr (KIND == kAllValues) {
            // The halves of the wavefront hold every other four vectors of a query; they change hands until a lane has eight that
            // follow each other, 16 bytes a store, whole lines by the tile's end.  (Bound by the products: 10,000 x 1M x 768 with 20 GB
            // stored 17.6 ms, 875 TFLOP/s.)
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                const int64_t q = q0 + 64 * wc + 32 * cb + l32;
                uint16_t *const to = out + (q < n_queries ? q : 0) * id0 + vt + 128 * wr + 8 * half;
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    uint32_t w[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        w[j] = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)acc[rb][cb][2 * j]) |
                               (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)acc[rb][cb][2 * j + 1]) << 16;
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        const auto a = __builtin_amdgcn_permlane32_swap(w[4 * p], w[4 * p + 2], false, false);
                        const auto b = __builtin_amdgcn_permlane32_swap(w[4 * p + 1], w[4 * p + 3], false, false);
                        if (q < n_queries) *reinterpret_cast<uint4 *>(to + 32 * rb + 16 * p) = make_uint4(a[0], b[0], a[1], b[1]);
                    }
                }
            }
        } else if constexpr (!EMIT) {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                    for (int r = 0; r < 16; ++r) top[cb][rb] = fmaxf(top[cb][rb], acc[rb][cb][r]);  // (whole tiles only)
        } else {
            if (vt + TR > v_end) {  // the strip's last tile repeats its last row
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    const int left = (int)(v_end - v_lane) - 32 * rb;  // rows of the strip from this lane's first on
#pragma unroll
                    for (int r = 0; r < 16; ++r)
#pragma unroll
                        for (int cb = 0; cb < CB; ++cb)
                            if (8 * (r >> 2) + (r & 3) >= left) acc[rb][cb][r] = -__builtin_inff();
                }
            }
            // A value is out if it is below thr (written so that a NaN is not).  Most blocks have none that is not; the
            // others are counted, get room with one atomic operation per lane and query for the whole tile, and the
            // comparisons are done again to store them.
            int hits[CB] = {0, 0};
            uint32_t some = 0;  // bit RB * cb + rb: a lane has one in this block
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    uint64_t any = 0;
#pragma unroll
                    for (int r = 0; r < 16; ++r) any |= __builtin_amdgcn_ballot_w64(!(acc[rb][cb][r] < thr[cb]));
                    if (any) {
                        some |= 1u << (RB * cb + rb);
                        float limit = thr[cb];
                        asm volatile("" : "+v"(limit));
#pragma unroll
                        for (int r = 0; r < 16; ++r) hits[cb] += !(acc[rb][cb][r] < limit);
                    }
                }
            if (some == 0) return;
            int at[CB];
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                const int64_t q = q0 + 64 * wc + 32 * cb + l32;
                at[cb] = hits[cb] && q < n_queries ? atomicAdd(&count[q], hits[cb]) : kFound;
            }
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                uint64_t *const dst = found + (q0 + 64 * wc + 32 * cb + l32) * kFound;
                float limit = thr[cb];
                asm volatile("" : "+v"(limit));  // compared again: 64 masks kept from above would not fit the scalar registers
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    if (((some >> (RB * cb + rb)) & 1) == 0) continue;
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const float value = acc[rb][cb][r];  // (a bit cast of a vector's element takes its first one)
                        const bool hit = !(value < limit);
                        if (__builtin_amdgcn_ballot_w64(hit) == 0) continue;
                        if (hit && at[cb] < kFound) {
                            const uint32_t id = (uint32_t)(id0 + v_lane) + (32 * rb + 8 * (r >> 2) + (r & 3));
                            dst[at[cb]++] = ((uint64_t)__builtin_bit_cast(uint32_t, value) << 32) | id;
                        }
                    }
                }
            }
        }
    };
    auto tile = [&](auto first, int64_t vt) __attribute__((always_inline)) {
        constexpr int P = decltype(first)::value;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[rb][cb][r] = 0.0f;
        for (int kt = 0; kt < kp2; kt += 2 * KT) {
            stage(std::integral_constant<int, P>{}, vt, kt);
            if (kt + KT < kp2) stage(std::integral_constant<int, P ^ 1>{}, vt, kt + KT);
        }
        fold(vt);
    };
    // the stage after a tile's last one goes into the other buffers: with an odd number of stages every second tile
    // starts from the second ones
    const bool odd = (kp2 / KT) & 1;
    for (int64_t vt = v_begin; vt < v_end;) {
        tile(std::integral_constant<int, 0>{}, vt);
        vt += TR;
        if (odd && vt < v_end) {
            tile(std::integral_constant<int, 1>{}, vt);
            vt += TR;
        }
    }
    if constexpr (KIND == kSampleMaxima) {
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            const int64_t q = q0 + 64 * wc + 32 * cb + l32;
            if (q < n_queries)
#pragma unroll
                for (int rb = 0; rb < RB; ++rb)
                    gmax[q * ((int64_t)n_strips * kGroupsPerStrip) + strip * kGroupsPerStrip + (wr * 2 + half) * RB + rb] =
                        top[cb][rb];
        }
    }
}

// What the sample tells of a query, from the k-th largest of its groups' maxima.  The queries that expect more than `most`
// vectors are counted in vmax.
__global__ __launch_bounds__(256) void bound_kernel(const float *__restrict__ gmax, int groups, int k, int64_t n_queries,
                                                    const RowStat *__restrict__ qstat, uint32_t *__restrict__ vmax,
                                                    int dim, int l2, float rows_per_sample_row, float most,
                                                    Sampled *__restrict__ bound, int32_t *__restrict__ count) {
    const int64_t q = (int64_t)blockIdx.x * 4 + threadIdx.x / kWave;
    if (q >= n_queries) return;
    const int lane = threadIdx.x & (kWave - 1);
    constexpr int PER = kMaxGroups / kWave;
    float top[PER];
    uint32_t key[PER];  // largest value first
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int g = lane + kWave * j;
        top[j] = g < groups ? gmax[q * groups + g] : -__builtin_inff();
        key[j] = ~vl_float_key(top[j] == top[j] ? top[j] : -__builtin_inff());  // a NaN bounds nothing
    }
    uint32_t kth = 0xFFFFFFFFu;
    for (int i = 0; i < k; ++i) {
        uint32_t mine = key[0];
#pragma unroll
        for (int j = 1; j < PER; ++j) mine = key[j] < mine ? key[j] : mine;
        kth = wave_min_u32(mine);
        // one of the groups that hold it is taken
        const uint64_t owners = __ballot(mine == kth);
        if (lane == __builtin_ctzll(owners)) {
            bool taken = false;
#pragma unroll
            for (int j = 0; j < PER; ++j)
                if (!taken && key[j] == kth) {
                    key[j] = 0xFFFFFFFFu;
                    taken = true;
                }
        }
    }
    const RowStat table = table_stat(vmax);
    const float error = value_error(qstat[q], table, dim, l2 != 0);
    float t = vl_key_float(~kth) - error;
    if (!l2) t = fminf(t, 1.0f - 1e-6f);  // values of 1 and more are one distance, 0
    // How many vectors will not be out: their rows of the sample lie in any group with the same chance, so a share of
    // exp(-m / groups) of the groups holds none of m such rows.
    const float limit = t - error;
    int without = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int g = lane + kWave * j;
        without += __popcll(__ballot(g < groups && top[j] < limit));
    }
    const float vectors = -(float)groups * logf((float)without / (float)groups) * rows_per_sample_row;  // infinite if none is without
    if (lane == 0) {
        bound[q] = Sampled{t, vectors, error};  // (no bound: no group is without)
        count[q] = 0;
        if (!(vectors <= most)) atomicAdd(vmax + (blockIdx.x & (kStripes - 1)) * kStripeWords + 2, 1u);
    }
}

__global__ void filter_clear_kernel(uint32_t *__restrict__ vmax, int64_t n, int32_t *__restrict__ left) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) vmax[i] = 0;
    if (i == 0 && left) left[0] = 0;
}

// Appends the queries with more candidates than a buffer holds to the list that the tiles take, in order, and gives their
// places the bound they start from.  One workgroup: it is the only one to touch the list.  (A place for each from an atomic
// counter took 8 ns a query where all were left.)
constexpr int kLeftThreads = 1024;
__global__ __launch_bounds__(kLeftThreads) void left_kernel(const int32_t *__restrict__ count, int n, int q_first,
                                                            int32_t *__restrict__ left, uint32_t *__restrict__ tile_bound) {
    constexpr int kWaves = kLeftThreads / kWave;
    __shared__ int part[2][kWaves];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    int have = left[0];
    for (int base = 0, round = 0; base < n; base += kLeftThreads, round ^= 1) {
        const int q = base + tid;
        const bool mine = q < n && count[q] > kFound;
        const uint64_t all = __ballot(mine);
        if (lane == 0) part[round][wave] = __popcll(all);
        __syncthreads();
        int at = have + __popcll(all & ((1ull << lane) - 1));
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const int theirs = part[round][w];
            have += theirs;
            if (w < wave) at += theirs;
        }
        if (mine) {
            left[1 + at] = q_first + q;
            tile_bound[at] = 0x7F800000u;
        }
    }
    if (tid == 0) left[0] = have;
}

// The dot products of up to 8 NG rows with the query, one row per lane: the products of knn_tile_kernel one fused
// multiply-add after the other, as its matrix instructions form them (element x of the two chunks of a pair, then y, z, w).
// The query row is the same for all lanes.  Rows come in lines of 32 columns, eight lanes to a line, and change hands in LDS
// (8 KB a wavefront, a chunk's place as in the tiles' operands): read by its own lane, a row costs a cycle of the address
// unit per 16 bytes (10,000 queries with some 950 rows each to evaluate at 32,768 x 768: 6.7 ms a call, 4.5 this way, which
// is 7.5 TB/s of rows).  Eight loads per lane are on their way whatever the number of rows, 8 / NG lines of each.
template <int NG>
__device__ __forceinline__ float dots_in_tile_order(const float *__restrict__ vectors, const int32_t *ids, int n,
                                                    const float *__restrict__ q, int dim, float4 *buf) {
    constexpr int D = 8 / NG;
    const int lane = threadIdx.x & (kWave - 1), c = lane & 7;
    const float *src[NG];
    int to[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        const int r = 8 * g + (lane >> 3);
        src[g] = vectors + (int64_t)ids[min(r, n - 1)] * dim + 4 * c;
        to[g] = r * CH + (c ^ swz(r));
    }
    const int own = lane & (8 * NG - 1);
    const float4 *const mine = buf + own * CH;
    const int lines = (dim + 31) / 32;
    float4 x[8];
    auto load = [&](int l0) {
#pragma unroll
        for (int d = 0; d < D; ++d)
#pragma unroll
            for (int g = 0; g < NG; ++g)
                if (8 * g < n && 32 * (l0 + d) + 4 * c < dim) x[d * NG + g] = *reinterpret_cast<const float4 *>(src[g] + 32 * (l0 + d));
    };
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    load(0);
    float s = 0.0f;
    auto pair = [&](const float4 &a, const float4 &b, const float *p) {
        s = fmaf(a.x, p[0], s); s = fmaf(b.x, p[4], s);
        s = fmaf(a.y, p[1], s); s = fmaf(b.y, p[5], s);
        s = fmaf(a.z, p[2], s); s = fmaf(b.z, p[6], s);
        s = fmaf(a.w, p[3], s); s = fmaf(b.w, p[7], s);
    };
    for (int l0 = 0; l0 < lines; l0 += D) {
#pragma unroll
        for (int d = 0; d < D; ++d)
#pragma unroll
            for (int g = 0; g < NG; ++g)
                if (d == 0 || l0 + d < lines) buf[d * 8 * NG * CH + to[g]] = x[d * NG + g];
        __builtin_amdgcn_wave_barrier();
        if (l0 + D < lines) load(l0 + D);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int left = dim - 32 * (l0 + d);  // columns
            const float *const p = q + 32 * (l0 + d);
            const float4 *const line = mine + d * 8 * NG * CH;
            if (left >= 32) {
                float4 a[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) a[i] = line[i ^ swz(own)];
#pragma unroll
                for (int i = 0; i < 4; ++i) pair(a[2 * i], a[2 * i + 1], p + 8 * i);
            } else {
                for (int i = 0; 8 * i < left; ++i) {
                    const float4 a = line[(2 * i) ^ swz(own)];
                    if (8 * i + 4 == left) {  // a last chunk on its own
                        s = fmaf(a.x, p[8 * i], s); s = fmaf(a.y, p[8 * i + 1], s); s = fmaf(a.z, p[8 * i + 2], s); s = fmaf(a.w, p[8 * i + 3], s);
                    } else {
                        pair(a, line[(2 * i + 1) ^ swz(own)], p + 8 * i);
                    }
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    return s;
}

// The k-th smallest of up to 64 values in LDS, a lane each: four values are looked at together (those past the last are not
// counted).  Bit by bit, as below, is 32 steps that wait for each other.
__device__ __forceinline__ uint32_t kth_of_a_few(const uint4 *values, int n, int k) {
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t mine = reinterpret_cast<const uint32_t *>(values)[min(lane, n - 1)];
    int below = 0, same = 0;
    for (int j = 0; 4 * j < n; ++j) {
        const uint4 x = values[j];
        below += (x.x < mine) + (4 * j + 1 < n && x.y < mine) + (4 * j + 2 < n && x.z < mine) + (4 * j + 3 < n && x.w < mine);
        same += (x.x == mine) + (4 * j + 1 < n && x.y == mine) + (4 * j + 2 < n && x.z == mine) + (4 * j + 3 < n && x.w == mine);
    }
    return (uint32_t)__builtin_amdgcn_readlane((int)mine, __builtin_ctzll(__builtin_amdgcn_ballot_w64(below < k && k <= below + same)));
}

// The k-th smallest of n values in LDS, 1 <= k <= n <= kFound, bit by bit; each wavefront finds it for itself.
template <int PER>
__device__ __forceinline__ uint32_t kth_of(const uint32_t *values, int n, int k) {
    const int lane = threadIdx.x & (kWave - 1);
    uint32_t v[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) v[j] = kWave * j + lane < n ? values[kWave * j + lane] : 0xFFFFFFFFu;
    uint32_t at = 0;
    for (uint32_t bit = 1u << 31; bit; bit >>= 1) {
        const uint32_t mid = at | bit;
        int below = 0;
#pragma unroll
        for (int j = 0; j < PER; ++j) below += __popcll(__builtin_amdgcn_ballot_w64(v[j] < mid));
        if (below < k) at = mid;
    }
    return at;
}
__device__ __forceinline__ uint32_t kth_smallest(const uint32_t *values, int n, int k) {
    if (n <= kWave) return kth_of_a_few(reinterpret_cast<const uint4 *>(values), n, k);
    if (n <= 4 * kWave) return kth_of<4>(values, n, k);
    if (n <= 16 * kWave) return kth_of<16>(values, n, k);
    return kth_of<kFound / kWave>(values, n, k);
}

// One workgroup per query.  The sample's bound let through several times k candidates; the k-th best value among all of
// them bounds the k-th best float32 value far better, so most are dropped before their rows are fetched (at 1,000 queries
// x 32,768 x 1,536, k = 16: 350 candidates, 390 us when all were evaluated).  What is left is evaluated, and those not
// above the k-th best distance are ranked.
// A few candidates with rows of up to so many columns are all evaluated at once: the bound on them would wait for LDS longer
// than their rows take (10,000 queries with 20 candidates of 64 columns each: 57.8 us with it, 44.5 without).
constexpr int kShortRow = 128;
template <bool L2, int THREADS>
__global__ __launch_bounds__(THREADS) void finish_kernel(const float *__restrict__ queries,
                                                         const float *__restrict__ vectors, int dim, int k,
                                                         const int32_t *__restrict__ count,
                                                         const uint64_t *__restrict__ found,
                                                         const RowStat *__restrict__ qstat,
                                                         const uint32_t *__restrict__ vmax, int slabs,
                                                         const float *__restrict__ q_norm,
                                                         const float *__restrict__ v_norm, int64_t q_first,
                                                         int32_t *__restrict__ ids_out, float *__restrict__ d_out) {
    constexpr int kWaves = THREADS / kWave;
    __shared__ float4 buf[kWaves][kWave * CH];
    __shared__ __align__(16) uint32_t values[kFound];  // of the pass, smallest is best; then the distances, as keys
    __shared__ int32_t ids[kFound];
    __shared__ int n_s, n_keys_s;
    uint64_t *const keys = reinterpret_cast<uint64_t *>(&buf[0][0]);
    static_assert(sizeof(buf) >= kFound * sizeof(uint64_t), "room for all keys");
    const int64_t q = q_first + blockIdx.x;
    const int tid = threadIdx.x;
    const int n = count[q];
    if (n > kFound) return;  // uniform; left to the tiles
    if (tid == 0) {
        n_s = 0;
        n_keys_s = 0;
    }
    const uint64_t own = tid < n ? found[q * kFound + tid] : 0;
    int left = n;
    if (n <= kWave && dim <= kShortRow) {
        if (tid < n) ids[tid] = (int32_t)(uint32_t)own;
        __syncthreads();
    } else {
        if (tid < n) values[tid] = ~vl_float_key(__builtin_bit_cast(float, (uint32_t)(own >> 32)));
        for (int i = tid + THREADS; i < n; i += THREADS) values[i] = ~vl_float_key(__builtin_bit_cast(float, (uint32_t)(found[q * kFound + i] >> 32)));
        RowStat table = {0.0f, 0.0f};
        for (int s = 1; s <= slabs; ++s) {
            const RowStat one = table_stat(vmax + (int64_t)s * kStripes * kStripeWords);
            table.resid = fmaxf(table.resid, one.resid);
            table.norm = fmaxf(table.norm, one.norm);
        }
        __syncthreads();
        float least = -__builtin_inff();
        if (n > k) {
            const float error = value_error(qstat[q], table, dim, L2);
            least = vl_key_float(~kth_smallest(values, n, k)) - error;
            if (!L2) least = fminf(least, 1.0f - 1e-6f);  // values of 1 and more are one distance, 0
            least -= error;
            if (!L2 && least <= -0.999f) least = -__builtin_inff();
        }
        for (int i = tid; i < n; i += THREADS)
            if (!(vl_key_float(~values[i]) < least)) ids[atomicAdd(&n_s, 1)] = (int32_t)(uint32_t)(i == tid ? own : found[q * kFound + i]);
        __syncthreads();
        left = __builtin_amdgcn_readfirstlane(n_s);
    }
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    for (int base = 0; base < left; base += THREADS) {
        // the same number of rows for each wavefront
        const int rows = min(left - base, THREADS), per = (rows + kWaves - 1) / kWaves;
        const int first = base + wave * per, mine = min(per, base + rows - first);
        if (mine <= 0) continue;
        float s;
        auto dots = [&](auto groups) {
            return dots_in_tile_order<decltype(groups)::value>(vectors, ids + first, mine, queries + q * dim, dim, buf[wave]);
        };
        if (mine <= 8) s = dots(std::integral_constant<int, 1>{});
        else if (mine <= 16) s = dots(std::integral_constant<int, 2>{});
        else if (mine <= 32) s = dots(std::integral_constant<int, 4>{});
        else s = dots(std::integral_constant<int, 8>{});
        const int i = first + (tid & (kWave - 1));
        if (i < first + mine) {
            const int32_t id = ids[i];
            values[i] = (uint32_t)(vl_make_key(id, tile_distance<L2>(s, L2 ? q_norm[q] : 0.0f, L2 ? v_norm[id] : 0.0f)) >> 32);
        }
    }
    __syncthreads();
    int n_keys = left;
    if (left <= kWave) {  // a few are ranked as they are
        if (tid < left) keys[tid] = ((uint64_t)values[tid] << 32) | (uint32_t)ids[tid];
        __syncthreads();
    } else {
        const uint32_t last = kth_smallest(values, left, k);
        for (int i = tid; i < left; i += THREADS)
            if (values[i] <= last) keys[atomicAdd(&n_keys_s, 1)] = ((uint64_t)values[i] << 32) | (uint32_t)ids[i];
        __syncthreads();
        n_keys = __builtin_amdgcn_readfirstlane(n_keys_s);
    }
    for (int i = tid; i < n_keys || i < k; i += THREADS) {
        if (i >= n_keys) {  // fewer vectors than asked for
            ids_out[q * k + i] = VL_MAXINT;
            d_out[q * k + i] = VL_MAXFLOAT;
            continue;
        }
        const uint64_t key = keys[i];
        int rank = 0;
        for (int j = 0; j < n_keys; ++j) rank += keys[j] < key;  // keys are unique
        if (rank < k) {
            ids_out[q * k + rank] = vl_key_id(key);
            d_out[q * k + rank] = vl_key_dist(key);
        }
    }
}

int64_t compute_units() {
    static const int64_t n = [] {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
            cus = 256;
        return (int64_t)cus;
    }();
    return n;
}

// strips of whole tiles for q_blocks query blocks on one workgroup per compute unit: the count (at most `most`) whose
// last round of workgroups ends first; a strip more costs an eighth of a tile (its start-up)
int64_t strips_for(int64_t q_blocks, int64_t tiles, int64_t most) {
    int64_t best = 1, best_cost = -1;
    for (int64_t s = 1; s <= most && s <= tiles; ++s) {
        const int64_t len = (tiles + s - 1) / s;
        if ((tiles + len - 1) / len != s) continue;
        const int64_t rounds = (q_blocks * s + compute_units() - 1) / compute_units();
        const int64_t cost = rounds * (8 * len + 1);
        if (best_cost < 0 || cost < best_cost) {
            best_cost = cost;
            best = s;
        }
    }
    return best;
}

inline int64_t align256(int64_t x) { return (x + 255) & ~255ll; }
inline int64_t gcd(int64_t a, int64_t b) { return b ? gcd(b, a % b) : a; }

}  // namespace

bool vl_knn_filter_plan(int64_t n_queries, int64_t n_vectors, int64_t dim, int64_t k, bool l2, KnnFilterPlan *p) {
    if (n_vectors < 4096 || dim > 8192) return false;
    p->kp = (dim + (l2 ? 3 : 0) + 63) / 64 * 64;
    const int64_t tiles = n_vectors / TR;
    // The sample: a sixteenth of the table (an eighth for long lists, whose expected number of candidates, k times the
    // share's inverse and half as much again for E, would come near kFound) and 32 tiles at least: a candidate costs as much
    // as some hundred products of 64 columns (32,768 entry points x 64 columns: 16 tiles 298 us, 32 tiles 242 us).
    int64_t sample = tiles / (k > 10 ? 8 : 16);
    if (sample < 32) sample = tiles / 2 < 32 ? (tiles + 1) / 2 : 32;
    p->sample_rows = sample * TR;
    p->sample_stride = p->sample_rows * 618 / 1000 | 1;
    while (gcd(p->sample_stride, p->sample_rows) != 1) p->sample_stride += 2;
    const int64_t q_blocks = (n_queries + TR - 1) / TR;
    int64_t strips = strips_for(q_blocks, sample, kMaxGroups / kGroupsPerStrip);
    // enough groups that the k-th largest maximum is close to the k-th best of the sample
    const int64_t least = sample < 16 ? sample : 16;
    if (strips < least) strips = least;
    const int64_t len = (sample + strips - 1) / strips;
    strips = (sample + len - 1) / len;
    p->sample_strips = (int)strips;
    p->groups = (int)(strips * kGroupsPerStrip);
    p->slab_rows = (2ll << 30) / (p->kp * 2) / TR * TR;
    if (p->slab_rows < p->sample_rows) p->slab_rows = p->sample_rows;
    if (p->slab_rows > n_vectors) p->slab_rows = n_vectors;
    // On full batches the tiles take 0.0163 ps per product and 0.14 ps per place of their lists for a vector, a candidate
    // 40 ps and 0.4 ps a column, and the pass, which a query left to the tiles saves as well, 0.002 ps per product.  A guess
    // somewhat above what the buffer holds is still tried (4,000 queries with 2,000 candidates each at 500,000 x 384: 4.5 ms,
    // with the tiles 12.8).
    const double even = (double)n_vectors * (0.014 * (double)dim + 0.14 * (double)k) / (40.0 + 0.4 * (double)dim);
    p->most = (int)(even < kMostExpected ? even : kMostExpected);
    int64_t o = 0;
    p->off_q16 = o; o = align256(o + n_queries * p->kp * 2);
    p->off_v16 = o; o = align256(o + p->slab_rows * p->kp * 2);
    p->off_qstat = o; o = align256(o + n_queries * (int64_t)sizeof(RowStat));
    p->off_gmax = o; o = align256(o + n_queries * p->groups * 4);
    p->off_bound = o; o = align256(o + n_queries * (int64_t)sizeof(Sampled));
    p->off_count = o; o = align256(o + n_queries * 4);
    p->off_found = o; o = align256(o + n_queries * kFound * 8);
    const int64_t slabs = (n_vectors + p->slab_rows - 1) / p->slab_rows;
    p->off_vmax = o; o = align256(o + (slabs + 1) * kStripes * kStripeWords * 4);
    p->bytes = o;
    return true;
}

int vl_knn_filter(const KnnFilterPlan &p, const float *queries, int64_t n_queries, const float *vectors, int64_t n_vectors,
                  int64_t dim, int64_t k, bool l2, float *q_norm, float *v_norm, int64_t q_first, int32_t *left,
                  uint32_t *tile_bound, char *ws, int32_t *ids_out, float *dists_out, hipStream_t st) {
    __bf16 *q16 = (__bf16 *)(ws + p.off_q16), *v16 = (__bf16 *)(ws + p.off_v16);
    RowStat *qstat = (RowStat *)(ws + p.off_qstat);
    float *gmax = (float *)(ws + p.off_gmax);
    Sampled *bound = (Sampled *)(ws + p.off_bound);
    int32_t *count = (int32_t *)(ws + p.off_count);
    uint64_t *found = (uint64_t *)(ws + p.off_found);
    uint32_t *vmax = (uint32_t *)(ws + p.off_vmax);
    const int kp = (int)p.kp, kp2 = kp / 2;
    const int64_t slabs = (n_vectors + p.slab_rows - 1) / p.slab_rows;
    const int64_t n_words = (slabs + 1) * kStripes * kStripeWords;
    const size_t smem = 4 * TR * KT * sizeof(float);
    auto allow = [&]() -> hipError_t {
        const hipError_t e = vl_allow_lds(pass_kernel<kSampleMaxima>, smem);
        return e == hipSuccess ? vl_allow_lds(pass_kernel<kCandidates>, smem) : e;
    };
    VL_HIP(allow());
    hipLaunchKernelGGL(filter_clear_kernel, dim3((unsigned)((n_words + 255) / 256)), dim3(256), 0, st, vmax,
                       n_words, q_first == 0 ? left : nullptr);
    const SampleRows sample{p.sample_rows, n_vectors, p.sample_stride};
    auto prepare = [&](auto kernel, const float *rows, int64_t n, int extra, __bf16 *out, float *norm2, RowStat *stat, uint32_t *top) {
        const int64_t blocks = (n + 3) / 4 < 2048 ? (n + 3) / 4 : 2048;
        hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), 0, st, rows, n, (int)dim, kp, sample, l2 ? extra : 0, out, norm2,
                           stat, top);
    };
    const int64_t q_blocks = (n_queries + TR - 1) / TR;
    int64_t q_group = (2ll << 20) / (TR * p.kp * 2);  // about 2 MB of query rows in one L2
    q_group = q_group < 1 ? 1 : (q_group > 8 ? 8 : q_group);
    auto pass = [&](bool emit, int64_t rows, int64_t strips, const uint32_t *top, int64_t id0) {
        const int64_t tiles = (rows + TR - 1) / TR;
        const int64_t len = (tiles + strips - 1) / strips * TR;
        const unsigned blocks = (unsigned)((q_blocks * strips + 7) / 8 * 8);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kThreads), smem, st, (const float *)q16, n_queries,
                               (const float *)v16, rows, kp2, len, (int)strips, (int)q_blocks, (int)q_group, gmax, bound,
                               qstat, top, vmax, (float)p.most, (int)dim, l2 ? 1 : 0, id0, count, found, nullptr);
        };
        if (emit) go(pass_kernel<kCandidates>);
        else go(pass_kernel<kSampleMaxima>);
    };
    prepare(prepare_kernel<false>, queries, n_queries, 1, q16, l2 ? q_norm : nullptr, qstat, nullptr);
    prepare(prepare_kernel<true>, vectors, p.sample_rows, 2, v16, nullptr, nullptr, vmax);
    VL_LAUNCH_CHECK("knn prepare_kernel");
    pass(false, p.sample_rows, p.sample_strips, vmax, 0);
    VL_LAUNCH_CHECK("knn pass_kernel (sample)");
    hipLaunchKernelGGL(bound_kernel, dim3((unsigned)((n_queries + 3) / 4)), dim3(256), 0, st, gmax, p.groups, (int)k,
                       n_queries, qstat, vmax, (int)dim, l2 ? 1 : 0, (float)n_vectors / (float)p.sample_rows, (float)p.most, bound,
                       count);
    VL_LAUNCH_CHECK("knn bound_kernel");
    for (int64_t s = 0; s < slabs; ++s) {
        const int64_t r0 = s * p.slab_rows;
        const int64_t rows = n_vectors - r0 < p.slab_rows ? n_vectors - r0 : p.slab_rows;
        prepare(prepare_kernel<false>, vectors + r0 * dim, rows, 2, v16, l2 ? v_norm + r0 : nullptr, nullptr, vmax + (s + 1) * kStripes * kStripeWords);
        pass(true, rows, strips_for(q_blocks, (rows + TR - 1) / TR, 1024), vmax + (s + 1) * kStripes * kStripeWords, r0);
        VL_LAUNCH_CHECK("knn pass_kernel (filter)");
    }
    for (int64_t q0 = 0; q0 < n_queries; q0 += kMaxBlocks) {
        const dim3 grid((unsigned)(n_queries - q0 < kMaxBlocks ? n_queries - q0 : kMaxBlocks));
        auto go = [&](auto kernel, int threads) {
            hipLaunchKernelGGL(kernel, grid, dim3((unsigned)threads), 0, st, queries, vectors, (int)dim, (int)k, count, found,
                               qstat, vmax, (int)slabs, q_norm, v_norm, q0, ids_out, dists_out);
        };
        if (n_queries <= kFinishWide) l2 ? go(finish_kernel<true, 512>, 512) : go(finish_kernel<false, 512>, 512);
        else l2 ? go(finish_kernel<true, 128>, 128) : go(finish_kernel<false, 128>, 128);
    }
    VL_LAUNCH_CHECK("knn finish_kernel");
    hipLaunchKernelGGL(left_kernel, dim3(1), dim3(kLeftThreads), 0, st, count, (int)n_queries, (int)q_first, left, tile_bound);
    VL_LAUNCH_CHECK("knn left_kernel");
    return VL_OK;
}

// ---- all products of a call's queries and vectors, for the beam step (near_products.h) ----

namespace {

// Rows rounded to bfloat16 and padded with zeros to kp columns and `padded` rows; a wavefront a row.  The queries in their order,
// the vectors in the order of PairColumns.
template <bool QUERIES>
__global__ __launch_bounds__(256) void near_prepare_kernel(const float *__restrict__ rows, int64_t n, int64_t padded, int dim, int kp,
                                                           __bf16 *__restrict__ out, NearQuery *__restrict__ queries,
                                                           uint32_t *__restrict__ columns) {
    const int lane = threadIdx.x & (kWave - 1);
    for (int64_t i = (int64_t)blockIdx.x * 4 + threadIdx.x / kWave; i < padded; i += (int64_t)gridDim.x * 4) {
        const int64_t row = QUERIES ? i : PairColumns(n).vector_at(i);
        const bool real = row < n;
        const float4 *src = reinterpret_cast<const float4 *>(rows + (real ? row : 0) * dim);
        bf16x4 *dst = reinterpret_cast<bf16x4 *>(out + i * kp);
        float s = 0.0f, e2 = 0.0f;
        for (int c = lane; c < kp / 4; c += kWave) {
            float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
            if (real && c < dim / 4) x = src[c];
            const bf16x4 h = {(__bf16)x.x, (__bf16)x.y, (__bf16)x.z, (__bf16)x.w};
            const float a = x.x - (float)h[0], b = x.y - (float)h[1], d = x.z - (float)h[2], e = x.w - (float)h[3];
            s = fmaf(x.x, x.x, fmaf(x.y, x.y, fmaf(x.z, x.z, fmaf(x.w, x.w, s))));
            e2 = fmaf(a, a, fmaf(b, b, fmaf(d, d, fmaf(e, e, e2))));
            dst[c] = h;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            s += __shfl_xor(s, o);
            e2 += __shfl_xor(e2, o);
        }
        float resid = up(sqrtf(e2)), norm = up(sqrtf(s));
        if (!(resid < 1e18f)) resid = __builtin_inff();  // also NaN
        if (!(norm < 1e18f)) norm = __builtin_inff();
        if (lane != 0) continue;
        if constexpr (QUERIES) {
            // what near_bounds multiplies a vector's residual and norm with, the float32 roundings of both sums included
            const float sums = (float)dim * 2.4e-7f * (norm + resid);
            queries[i] = NearQuery{up(norm + resid) + sums, resid + sums};
        } else {
            columns[i] = half_bits_not_below(resid) | half_bits_not_below(norm) << 16;
        }
    }
}

}  // namespace

NearPlan vl_near_plan(int64_t n_queries, int64_t n_vectors, int64_t dim) {
    NearPlan p;
    p.kp = (dim + 63) / 64 * 64;
    p.columns = (PairColumns(n_vectors).count() + TR - 1) / TR * TR;
    int64_t o = 0;
    p.off_queries = o; o = align256(o + n_queries * (int64_t)sizeof(NearQuery));
    p.off_columns = o; o = align256(o + p.columns * 4);
    p.off_q16 = o; o = align256(o + n_queries * p.kp * 2);
    p.off_v16 = o; o = align256(o + p.columns * p.kp * 2);
    p.off_values = o; o = align256(o + n_queries * p.columns * 2);
    p.bytes = o;
    return p;
}

int vl_launch_near_products(const NearPlan &p, const float *queries, int64_t n_queries, const float *vectors, int64_t n_vectors,
                            int64_t dim, uint8_t *ws, hipStream_t st) {
    const size_t smem = 4 * TR * KT * sizeof(float);
    VL_HIP(vl_allow_lds(pass_kernel<kAllValues>, smem));
    __bf16 *const q16 = (__bf16 *)(ws + p.off_q16), *const v16 = (__bf16 *)(ws + p.off_v16);
    auto blocks_for = [](int64_t rows) { return dim3((unsigned)((rows + 3) / 4 < 4096 ? (rows + 3) / 4 : 4096)); };
    hipLaunchKernelGGL(near_prepare_kernel<true>, blocks_for(n_queries), dim3(256), 0, st, queries, n_queries, n_queries, (int)dim,
                       (int)p.kp, q16, (NearQuery *)(ws + p.off_queries), (uint32_t *)nullptr);
    hipLaunchKernelGGL(near_prepare_kernel<false>, blocks_for(p.columns), dim3(256), 0, st, vectors, n_vectors, p.columns, (int)dim,
                       (int)p.kp, v16, (NearQuery *)nullptr, (uint32_t *)(ws + p.off_columns));
    VL_LAUNCH_CHECK("near_prepare_kernel");
    const int64_t q_blocks = (n_queries + TR - 1) / TR, tiles = p.columns / TR, strips = strips_for(q_blocks, tiles, 1024);
    const int64_t len = (tiles + strips - 1) / strips * TR;
    int64_t q_group = (2ll << 20) / (TR * p.kp * 2);
    q_group = q_group < 1 ? 1 : (q_group > 8 ? 8 : q_group);
    hipLaunchKernelGGL(pass_kernel<kAllValues>, dim3((unsigned)((q_blocks * strips + 7) / 8 * 8)), dim3(kThreads), smem, st,
                       (const float *)q16, n_queries, (const float *)v16, p.columns, (int)p.kp / 2, len, (int)strips, (int)q_blocks,
                       (int)q_group, nullptr, nullptr, nullptr, nullptr, nullptr, 0.0f, (int)dim, 0, p.columns, nullptr, nullptr,
                       (uint16_t *)(ws + p.off_values));
    VL_LAUNCH_CHECK("pass_kernel (all values)");
    return VL_OK;
}
