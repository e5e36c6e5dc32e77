// Ball query, packed layout, over a hash table of cells (several clouds back to back, sorted cloud id per point).
//
// Space is cut into cells of 0.55 x 2.2 x 2.2 reaches (the reach: the radius and its rounding), and cell (ix, iy, iz) of a cloud
// belongs to bucket row(iy, iz, cloud) + ix of a table with 2 .. 4 buckets per support point, 131072 at least: the cells a ball touches are
// at most four runs (two values of iy, two of iz; three each within rounding of an edge) of four or five consecutive buckets.  No
// bounding box, no windows, no limit on a cloud's size: the launches in front of the queries clear the table, count the points
// per bucket (the atomic that counts hands out the point's place in its bucket), turn the counts into places, and put the points
// there as records (x, y, z, row).  Points of other cells that share a bucket fail the radius test or lie in another cloud's rows.
//
// A wavefront answers four queries, 16 lanes each, as wide as a row of the DPP network: a lane looks up a run, prefix sums
// over the 16 give the query's candidates, which are tested 16 at a time.  Hits are collected in LDS and ranked by row,
// which is the order a serial scan in index order that stops after nsample hits (cuda/src/ball_query_gpu.cu:54-95) meets them in.
// A query with more than 128 keeps the nsample lowest rows and goes on.  Where that scan itself is likely to end sooner than the
// walk - dense neighbourhoods -, or the query has more candidates than its cloud has rows, the wavefront scans, for all such queries of
// a cloud among its four at once; a query with many candidates is walked for by the whole wavefront.
//
// Measured against the walk over bins of windows (nn_grid.hip: windows of consecutive rows, each of which a query has to look
// into), whole calls, us: 53000 queries of four scenes of 20000 .. 100000 points 50 -> 42 (15 of them the queries, 37
// before; clearing 3, counting 13, places 4, records 7, against 17 for the windows' ordering), all 212000 of their points as queries 117 ->
// 61 (nsample 16, radius 0.04), 138 -> 75 (64, 0.1), 2300 -> 272 (64, 0.3: 60 points in a ball of a plane, which the walk over bins
// left to the scan); 300000 queries of 24 clouds 257 -> 133.  By radius in rooms of 8, nsample 16 / 64:
//     radius                       0.1                      0.3                      0.6                      1                        1.4                      2
//     53000 of 4 clouds, 212000    57 / 57 -> 44 / 46       275 / 830 -> 87 / 87     305 / 709 -> 210 / 305   164 / 461 -> 115 / 278   83 / 243 -> 73 / 177     54 / 131 -> 49 / 106
//     12500 of 1 cloud, 100000     32 / 33 -> 31 / 30       160 / 479 -> 55 / 57     176 / 309 -> 92 / 161    82 / 203 -> 72 / 140     46 / 116 -> 48 / 107     31 / 65 -> 32 / 64
//     50000 of 1 cloud, 100000     53 / 54 -> 36 / 38       415 / 1446 -> 95 / 97    313 / 750 -> 179 / 371   152 / 471 -> 110 / 269   85 / 253 -> 66 / 172     52 / 133 -> 46 / 100
//     17000 of 1 cloud, 200000     48 / 49 -> 44 / 45       525 / 794 -> 95 / 121    261 / 667 -> 153 / 263   85 / 275 -> 76 / 194     51 / 131 -> 49 / 116     37 / 76 -> 37 / 72
//     24000 of 12 clouds, 24000    29 / 31 -> 21 / 23       31 / 33 -> 23 / 24       43 / 45 -> 24 / 26       51 / 53 -> 30 / 31       45 / 62 -> 39 / 43       34 / 59 -> 34 / 51
//     9000 of 1 cloud, 9000        22 / 24 -> 20 / 20       24 / 25 -> 21 / 22       38 / 42 -> 28 / 27       47 / 80 -> 44 / 56       38 / 65 -> 40 / 73       30 / 49 -> 31 / 56
//     300000 of 24 clouds, 300000  153 / 151 -> 82 / 97     176 / 178 -> 90 / 96     402 / 442 -> 204 / 201   604 / 1491 -> 355 / 661  322 / 991 -> 242 / 612   183 / 549 -> 156 / 360
// What bounds it: the counting its atomics, the queries instruction issue - 690 vector instructions per wavefront, 170 per query
// with 16 hits each, of 1700 clocks a query before.
// Sorted neighbours (calls against the walk over bins that merged a sorted list, us): 212000 queries of the four scenes 188 -> 69 (16 slots, radius
// 0.04), 271 -> 85 (64, 0.1), 768 -> 366 (64, 0.3); an eighth of them 48 -> 37 and 67 -> 44.
// Cells of 1.1 and 0.28 reaches along x: the 300000 queries 96 and 94 us against 94, counting 15 and 13 against 13.
#include <algorithm>
#include <cmath>

#include "ball_scan.h"
#include "ball_table.h"
#include "cloud_rows.h"
#include "nn_grid.h"
#include "topk.h"

namespace {

constexpr int BT_THREADS = 256;
constexpr int BT_GROUP = 16;                       // lanes per query
constexpr int BT_QUERIES = TPK_WAVE / BT_GROUP;    // queries per wavefront
constexpr int BT_HITS = 2 * TPK_WAVE;              // hits a query holds when a step begins
constexpr int BT_KEPT = TPK_WAVE;                  // slots of a call whose queries may keep their lowest rows when they hold more
constexpr int BT_LONG = 128;                       // candidates from which on a query may be scanned for at once
constexpr float BT_MOST_HIT = 0.5f, BT_LEAST_HIT = 1.0f / 64; // of such a query's candidates in the ball, as far as nobody has looked
constexpr int BT_SAMPLES = 4;                      // of its candidates, per lane, that tell how many of them lie in the ball
// Candidates from which on a query's walk is the whole wavefront's, 64 a step (256: 53000 queries of 212000 points in rooms of 8, radius 0.3,
// 90 / 94 us instead of 87 / 87; 1024: 17000 of 200000, radius 1.4, 59 instead of 49), and hits it holds when a step begins.
constexpr int BT_ALONE = 768, BT_ALONE_HITS = BT_HITS + BT_GROUP - TPK_WAVE;
constexpr int BT_ALONE_AHEAD = 3;                  // steps of it whose candidates are requested together (2: 1 % slower)
constexpr int BT_HIT_STRIDE = BT_HITS + BT_GROUP + 4; // (the four queries of a wavefront read theirs at the same time: other banks)
constexpr int BT_COUNT_THREADS = 1024;
constexpr int BT_AHEAD = 2;                        // steps whose candidates are requested together (3: 300000 queries, radius 0.1, 87 / 110 us instead of 82 / 96)
// Points of a wavefront that share the buckets of four others, from which on a small array's workgroup counts in LDS first.  (Always: 9000 and
// 24000 points, radius 0.3 in rooms of 8, counting 6.2 and 6.7 us instead of 3.8 and 5; 2: 24000 points, radius 0.1 to 0.6, calls of 21 to 26 us
// 0.5 to 1.6 longer; never, see bt_count_kernel.)
constexpr int BT_SHARED = 4;
constexpr unsigned BT_NO_BUCKET = 0xffffffffu;
constexpr int BT_SCAN_THREADS = 1024;
constexpr int BT_CHUNK = BT_SCAN_THREADS * 4;      // buckets whose places one workgroup hands out
// Points of a counting workgroup: 256 below 65536 points, 512 below 131072, then 1024.  The more there are, the fewer atomics wait for each other
// where cells are full; the fewer, the more compute units share a small array.  48000 / 57000 points, radius 0.09: 5.9 / 6.2 us with 256, 7.2 / 7.5
// with 1024; 100000 points in a room of 8, radius 2: whole call 36 / 34 / 33 us; 212000, radius 0.05: 13.7 with 1024, 14 with 512.
constexpr int64_t BT_COUNT_MEDIUM = 65536, BT_COUNT_LARGE = 131072;
constexpr int BT_MOST_X = BT_CHUNK / 2;            // buckets of a run, at most: a run touches two chunks at most
constexpr float BT_WIDTH_X = 0.55f, BT_WIDTH_YZ = 2.2f; // of a cell, in reaches

struct CellScale
{
    float reach, inverse_x, inverse_yz;
};

__global__ void __launch_bounds__(BT_THREADS) bt_clear_kernel(int64_t quads, int4* table)
{
    const int64_t i = (int64_t)blockIdx.x * BT_THREADS + threadIdx.x;
    if (i < quads)
        table[i] = make_int4(0, 0, 0, 0);
}

__device__ __forceinline__ uint32_t bt_point_bucket(float x, float y, float z, int64_t cloud, const CellScale& scale, uint32_t part_mask)
{
    return bt_bucket(bt_row(bt_cell(y, scale.inverse_yz), bt_cell(z, scale.inverse_yz), cloud), bt_cell(x, scale.inverse_x), part_mask);
}

// counts: how many points every bucket holds; ranks: the place of every point among its bucket's.  Workgroups behind those of the
// points find the rows of every query's cloud.
// Bound by the atomics (16 to the nanosecond where they go to different buckets), which wait for each other where they do not, 20 to 60 ns
// each: the workgroup counts its own points in LDS first and sends one atomic per bucket.  212000 points of four scenes, radius 0.05: 13 us,
// and 13 with an atomic per point and lanes that share the wavefront's first bucket; 100000 points, radius 0.6 / 2 / 6 in a
// room of 8: 8 / 4 / 5 us instead of 30 / 130 / 530; a million points 56 instead of 65 and, radius 0.5, 33 instead of 154.  (Atomics at once unless a
// wavefront's points share the first one's bucket: 8 / 5 / 5 and 53.)
template <int COUNT_THREADS>
__global__ void __launch_bounds__(COUNT_THREADS)
    bt_count_kernel(int n, unsigned point_blocks, const float* __restrict__ x, const int64_t* __restrict__ batch_x, CellScale scale, uint32_t part_mask,
                    int* counts, int* __restrict__ ranks, int* __restrict__ placed, CloudRows rows)
{
    constexpr int SLOTS = 2 * COUNT_THREADS; // of the table in LDS: every point of the workgroup may need one
    __shared__ unsigned keys[SLOTS];
    __shared__ int shared_counts[SLOTS];
    if (blockIdx.x >= point_blocks)
    {
        cloud_rows_job(rows, static_cast<int64_t>(blockIdx.x - point_blocks) * (COUNT_THREADS / TPK_WAVE) + threadIdx.x / TPK_WAVE,
                       threadIdx.x & (TPK_WAVE - 1));
        return;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0)
        *placed = 0;
    const int i = blockIdx.x * COUNT_THREADS + threadIdx.x;
    const bool has = i < n;
    const int64_t at = has ? i : 0;
    const uint32_t bucket = bt_point_bucket(x[at * 3 + 0], x[at * 3 + 1], x[at * 3 + 2], batch_x[at], scale, part_mask);
    if constexpr (COUNT_THREADS < BT_COUNT_THREADS / 2)
    {
        // Small arrays: how many of a wavefront's points share the buckets of four of them?
        int sharing = 0;
#pragma unroll
        for (int probe = 0; probe < TPK_WAVE; probe += TPK_WAVE / 4)
        {
            const uint32_t of_probe = static_cast<uint32_t>(tpk_read_lane(static_cast<int>(bucket), probe));
            sharing += __builtin_popcountll(__ballot(has && bucket == of_probe));
        }
        if (__syncthreads_or(sharing >= 4 + BT_SHARED) == 0)
        {
            if (has)
                ranks[i] = atomicAdd(&counts[bucket], 1);
            return;
        }
    }
    for (int slot = threadIdx.x; slot < SLOTS; slot += COUNT_THREADS)
    {
        keys[slot] = BT_NO_BUCKET;
        shared_counts[slot] = 0;
    }
    __syncthreads();
    int slot = static_cast<int>(bucket % SLOTS), rank = 0;
    if (has)
    {
        for (;;)
        {
            const unsigned there = atomicCAS(&keys[slot], BT_NO_BUCKET, bucket);
            if (there == BT_NO_BUCKET || there == bucket)
                break;
            slot = (slot + 1) % SLOTS;
        }
        rank = atomicAdd(&shared_counts[slot], 1);
    }
    __syncthreads();
    for (int s = threadIdx.x; s < SLOTS; s += COUNT_THREADS)
        if (shared_counts[s] > 0)
            shared_counts[s] = atomicAdd(&counts[keys[s]], shared_counts[s]);
    __syncthreads();
    if (has)
        ranks[i] = shared_counts[slot] + rank;
}

// Counts -> first places, in place.  Every workgroup sums a chunk of the table and takes its range of places with one atomic: the
// chunks' ranges lie in no particular order, and a run of buckets that crosses from one chunk to the next is looked up as
// two.  chunk_ends: where a chunk's last bucket ends.
__global__ void __launch_bounds__(BT_SCAN_THREADS) bt_places_kernel(int4* table, int* __restrict__ chunk_ends, int* placed)
{
    __shared__ int waves[BT_SCAN_THREADS / TPK_WAVE];
    __shared__ int base;
    const int wave = threadIdx.x / TPK_WAVE, lane = threadIdx.x % TPK_WAVE;
    const int64_t at = (int64_t)blockIdx.x * BT_SCAN_THREADS + threadIdx.x;
    const int4 c = table[at];
    const int mine = c.x + c.y + c.z + c.w;
    const int before = wave_exclusive_sum(mine);
    if (lane == TPK_WAVE - 1)
        waves[wave] = before + mine;
    __syncthreads();
    if (wave == 0)
    {
        const int v = lane < BT_SCAN_THREADS / TPK_WAVE ? waves[lane] : 0;
        const int sum = wave_exclusive_sum(v);
        if (lane < BT_SCAN_THREADS / TPK_WAVE)
            waves[lane] = sum;
        if (lane == TPK_WAVE - 1)
        {
            base = atomicAdd(placed, sum + v);
            chunk_ends[blockIdx.x] = base + sum + v;
        }
    }
    __syncthreads();
    const int first = base + waves[wave] + before;
    table[at] = make_int4(first, first + c.x, first + c.x + c.y, first + c.x + c.y + c.z);
}

__global__ void __launch_bounds__(BT_THREADS)
    bt_records_kernel(int n, const float* __restrict__ x, const int64_t* __restrict__ batch_x, CellScale scale, uint32_t part_mask,
                      const int* __restrict__ table, const int* __restrict__ ranks, float4* __restrict__ records)
{
    const int i = blockIdx.x * BT_THREADS + threadIdx.x;
    if (i >= n)
        return;
    const float px = x[(int64_t)i * 3 + 0], py = x[(int64_t)i * 3 + 1], pz = x[(int64_t)i * 3 + 2];
    const uint32_t bucket = bt_point_bucket(px, py, pz, batch_x[i], scale, part_mask);
    records[table[bucket] + ranks[i]] = make_float4(px, py, pz, __int_as_float(i));
}

// (value of the row's lane L)
template <int L>
__device__ __forceinline__ int row_lane(int v)
{
    return __builtin_amdgcn_ds_swizzle(v, (L << 5) | 0x10); // and-mask 0x10, or-mask L: in every half wavefront, per row
}

// What hits are ordered by: their rows, or (SORTED) squared distance and then row - the 64 bits of a hit as they lie in LDS.
template <bool SORTED>
struct HitKey;
template <>
struct HitKey<false>
{
    using type = int;
    static constexpr type NONE = 0x7fffffff;
    static __device__ __forceinline__ type of(int2 hit) { return hit.x; }
    template <int BY>
    static __device__ __forceinline__ type turned(type v) // row_ror:BY
    {
        return __builtin_amdgcn_update_dpp(0, v, 0x120 + BY, 0xF, 0xF, true);
    }
    static __device__ __forceinline__ type from_lane(type v, int lane) { return tpk_read_lane(v, lane); }
};
template <>
struct HitKey<true>
{
    using type = u64;
    static constexpr type NONE = ~0ull;
    static __device__ __forceinline__ type of(int2 hit) { return static_cast<u64>(static_cast<unsigned>(hit.y)) << 32 | static_cast<unsigned>(hit.x); }
    template <int BY>
    static __device__ __forceinline__ type turned(type v)
    {
        return of(make_int2(HitKey<false>::turned<BY>(static_cast<int>(v)), HitKey<false>::turned<BY>(static_cast<int>(v >> 32))));
    }
    static __device__ __forceinline__ type from_lane(type v, int lane) { return read_lane_key(v, lane); }
};

// How many of the row's values are below `mine`, its own among them.
template <bool SORTED, int BY = 1>
__device__ __forceinline__ int rank_among_row(typename HitKey<SORTED>::type mine)
{
    if constexpr (BY == BT_GROUP)
        return 0;
    else
        return (HitKey<SORTED>::template turned<BY>(mine) < mine ? 1 : 0) + rank_among_row<SORTED, BY + 1>(mine);
}

// Puts the first cnt hits of every query of the wavefront (int2 (row, distance); cnt is the same in a query's 16 lanes) in ascending order;
// those that are not among the nsample lowest go.  (cnt 0: a query whose hits stay as they are.)  Up to 16 and 32 hits a query's own lanes rank them, one or two each; above, the
// whole wavefront ranks one query's after the other's by lane reads, three instructions per hit.
template <bool SORTED>
__device__ __forceinline__ void order_hits(int2* wave_hits, int cnt, int lane, int nsample)
{
    using K = HitKey<SORTED>;
    using Key = typename K::type;
    const int group = lane / BT_GROUP, sub = lane % BT_GROUP;
    int2* const hits = wave_hits + group * BT_HIT_STRIDE;
    const int most = rows_max(cnt);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (most <= BT_GROUP)
    {
        const int2 hit = hits[sub];
        const int rank = rank_among_row<SORTED>(sub < cnt ? K::of(hit) : K::NONE);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (sub < cnt && rank < nsample)
            hits[rank] = hit;
    }
    else if (most <= 2 * BT_GROUP)
    {
        const int2 hit0 = hits[sub], hit1 = hits[BT_GROUP + sub];
        const Key mine0 = K::of(hit0), mine1 = K::of(hit1);
        int rank0 = 0, rank1 = 0;
        for (int i = 0; i < most; ++i)
        {
            const Key other = i < cnt ? K::of(hits[i]) : K::NONE;
            rank0 += other < mine0 ? 1 : 0;
            rank1 += other < mine1 ? 1 : 0;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (sub < cnt && rank0 < nsample)
            hits[rank0] = hit0;
        if (BT_GROUP + sub < cnt && rank1 < nsample)
            hits[rank1] = hit1;
    }
    else
    {
        for (int g = 0; g < BT_QUERIES; ++g)
        {
            int2* const of_g = wave_hits + g * BT_HIT_STRIDE;
            const int count = tpk_read_lane(cnt, g * BT_GROUP);
            if (count == 0)
                continue;
            if (count <= TPK_WAVE)
            {
                const int2 hit = of_g[lane];
                const Key mine = lane < count ? K::of(hit) : K::NONE;
                int rank = 0;
                for (int i = 0; i < count; ++i)
                    rank += K::from_lane(mine, i) < mine ? 1 : 0;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                if (lane < count && rank < nsample)
                    of_g[rank] = hit;
                continue;
            }
            // (a query that is full: up to 144)
            constexpr int PER = 3;
            static_assert(PER * TPK_WAVE >= BT_HITS + BT_GROUP, "every hit has a register");
            int2 hit[PER];
            int rank[PER];
            if (lane < 4)
                of_g[count + lane] = make_int2(SORTED ? -1 : 0x7fffffff, -1); // (read four at a time; behind all hits)
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int j = 0; j < PER; ++j)
            {
                hit[j] = of_g[min(j * TPK_WAVE + lane, BT_HIT_STRIDE - 1)];
                rank[j] = 0;
            }
            for (int i = 0; i < count; i += 4)
            {
                Key other[4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    other[u] = K::of(of_g[i + u]);
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int j = 0; j < PER; ++j)
                        rank[j] += other[u] < K::of(hit[j]) ? 1 : 0;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int j = 0; j < PER; ++j)
                if (j * TPK_WAVE + lane < count && rank[j] < nsample)
                    of_g[rank[j]] = hit[j];
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// Whether a scan of the cloud in index order is likely to take less time than a walk over `candidates` more, for a query with
// about `hits` hits.  The scan meets nsample of them within rows * nsample / hits rows, 64 a step of `per_step` instructions; a step of the
// walk takes 45 for 16 candidates of each of four queries, or of 64 of one.  A scan's step counts 10 (9 for the test, 12 more where it holds hits)
// before the walk, and 25 after the first hits, when most of what is left of a walk is short.  (8 / 10 / 14 before the walk: 100000 points in a
// room of 8, 12500 queries, nsample 16, radius 0.6, 102 / 92 / 81 us; 64 slots, radius 1.4, 103 / 107 / 117; 300000 queries of 24 clouds, 64
// slots, radius 1.4, 562 / 612 / 757.)
constexpr float BT_SCAN_STEP = 10.0f, BT_SCAN_STEP_LATER = 25.0f;
__device__ __forceinline__ bool scan_is_shorter(float rows, float nsample, float hits, float candidates, float per_step)
{
    const float scan = fminf(rows, rows * nsample * __builtin_amdgcn_rcpf(hits)) * (per_step / TPK_WAVE);
    return candidates * (45.0f / (BT_GROUP * BT_QUERIES)) > scan;
}

// The support rows s0 .. s1 against those of the wavefront's four queries whose first lanes are set in `which`, as ball_scan_rows does
// for one: a step's rows are loaded once for all of them.  Hits go to a list in LDS, from there 64 at a time to the outputs: where balls are
// large most steps have a few, and two stores to memory and their addresses take three times the instructions (300000 queries of 24 rooms,
// radius 2, nsample 16 / 64: 181 / 440 us stored one by one, 151 / 330 this way).  A step tests its rows against all four at once, without
// looking which are done, so the last one's rows are tested by themselves (12500 queries of 100000 points, radius 1: 83 / 181 us -> 73 / 145).
__device__ __forceinline__ void bt_scan_rows(const float* __restrict__ x, int s0, int s1, unsigned long long which, float qx, float qy, float qz,
                                             float radius2, int nsample, int lane, int2* wave_hits, int64_t* __restrict__ idx4,
                                             float* __restrict__ dist4 TPK_WORK_PARAM)
{
    constexpr int BATCH = 4; // loads of four steps in flight (6: 3 % slower; the next four requested ahead: nothing)
    static_assert(2 * TPK_WAVE <= BT_HIT_STRIDE, "less than 64 hits wait in a query's list, and a step adds up to 64");
    float x4[BT_QUERIES], y4[BT_QUERIES], z4[BT_QUERIES];
    const unsigned slots = nsample;
    unsigned cnt[BT_QUERIES];
#pragma unroll
    for (int g = 0; g < BT_QUERIES; ++g)
    {
        x4[g] = to_vector_register(tpk_read_lane(qx, g * BT_GROUP));
        y4[g] = to_vector_register(tpk_read_lane(qy, g * BT_GROUP));
        z4[g] = to_vector_register(tpk_read_lane(qz, g * BT_GROUP));
        cnt[g] = which >> (g * BT_GROUP) & 1 ? 0 : slots;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const float none = __builtin_nanf("");
#pragma unroll
    for (int g = 0; g < BT_QUERIES; ++g)
        x4[g] = cnt[g] < slots ? x4[g] : none; // (no row is within reach of a query that is done)
    float px[BATCH], py[BATCH], pz[BATCH];
    auto load = [&](int base) __attribute__((always_inline)) {
        const float* __restrict__ const at = x + static_cast<int64_t>(base) * 3;
        const int last = s1 - 1 - base;
        if (last >= BATCH * TPK_WAVE - 1)
        {
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
            {
                const unsigned word = static_cast<unsigned>(lane) * 3u + u * (TPK_WAVE * 3u);
                px[u] = at[word + 0u];
                py[u] = at[word + 1u];
                pz[u] = at[word + 2u];
            }
        }
        else
        {
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
            {
                const int row = u * TPK_WAVE + lane;
                const unsigned word = static_cast<unsigned>(min(row, last)) * 3u;
                px[u] = row <= last ? at[word + 0u] : none;
                py[u] = at[word + 1u];
                pz[u] = at[word + 2u];
            }
        }
    };
    // Adds the hits of a step to a query's list and hands on 64 of them where it holds as many.
    auto keep = [&](bool hit, unsigned long long mask, int pos, float d, int2* list, unsigned& count, int64_t* its_idx, float* its_dist) __attribute__((always_inline)) {
        const unsigned waiting = count % TPK_WAVE, found = __builtin_popcountll(mask);
        if (hit)
            list[__builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(mask >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(mask), waiting))] =
                make_int2(pos, __float_as_int(d));
        count += found;
        if (waiting + found < TPK_WAVE)
            return;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const unsigned s = count / TPK_WAVE * TPK_WAVE - TPK_WAVE + lane;
        const int2 first = list[lane], behind = list[TPK_WAVE + lane];
        if (s < slots)
        {
            its_idx[s] = first.x;
            its_dist[s] = __int_as_float(first.y);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        list[lane] = behind;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    auto active = [&]() __attribute__((always_inline)) {
        return (cnt[0] < slots ? 1 : 0) + (cnt[1] < slots ? 1 : 0) + (cnt[2] < slots ? 1 : 0) + (cnt[3] < slots ? 1 : 0);
    };
    int base = s0;
    for (; base < s1 && active() > 1; base += BATCH * TPK_WAVE)
    {
        load(base);
#pragma unroll
        for (int u = 0; u < BATCH; ++u)
        {
            // (all four at once: a test has to wait for the test in front of it only where there are hits)
            float d[BT_QUERIES];
            unsigned long long mask[BT_QUERIES];
#pragma unroll
            for (int g = 0; g < BT_QUERIES; ++g)
            {
                d[g] = tpk_dist2(x4[g], y4[g], z4[g], px[u], py[u], pz[u]);
                TPK_WORK_ADD(1);
            }
#pragma unroll
            for (int g = 0; g < BT_QUERIES; ++g)
                mask[g] = __ballot(d[g] <= radius2);
            if (((mask[0] | mask[1]) | (mask[2] | mask[3])) == 0)
                continue; // (most steps of a long scan)
            const int pos = base + u * TPK_WAVE + lane;
#pragma unroll
            for (int g = 0; g < BT_QUERIES; ++g)
            {
                if (mask[g] == 0)
                    continue;
                keep(d[g] <= radius2, mask[g], pos, d[g], wave_hits + g * BT_HIT_STRIDE, cnt[g], idx4 + g * slots, dist4 + g * slots);
                x4[g] = cnt[g] < slots ? x4[g] : none;
            }
        }
    }
    // The last one's rows, without the others' tests.
    if (base < s1 && active() == 1)
    {
        const int g = cnt[0] < slots ? 0 : cnt[1] < slots ? 1 : cnt[2] < slots ? 2 : 3;
        const float x1 = g < 2 ? (g == 0 ? x4[0] : x4[1]) : (g == 2 ? x4[2] : x4[3]), y1 = g < 2 ? (g == 0 ? y4[0] : y4[1]) : (g == 2 ? y4[2] : y4[3]),
                    z1 = g < 2 ? (g == 0 ? z4[0] : z4[1]) : (g == 2 ? z4[2] : z4[3]);
        unsigned count = g < 2 ? (g == 0 ? cnt[0] : cnt[1]) : (g == 2 ? cnt[2] : cnt[3]);
        for (; base < s1 && count < slots; base += BATCH * TPK_WAVE)
        {
            load(base);
            float d[BATCH];
            unsigned long long mask[BATCH];
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
            {
                d[u] = tpk_dist2(x1, y1, z1, px[u], py[u], pz[u]);
                TPK_WORK_ADD(1);
            }
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
                mask[u] = __ballot(d[u] <= radius2);
            if (((mask[0] | mask[1]) | (mask[2] | mask[3])) == 0)
                continue;
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
                if (mask[u] != 0 && count < slots)
                    keep(d[u] <= radius2, mask[u], base + u * TPK_WAVE + lane, d[u], wave_hits + g * BT_HIT_STRIDE, count, idx4 + g * slots, dist4 + g * slots);
        }
#pragma unroll
        for (int h = 0; h < BT_QUERIES; ++h)
            cnt[h] = h == g ? count : cnt[h];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int g = 0; g < BT_QUERIES; ++g)
        if (which >> (g * BT_GROUP) & 1)
            for (unsigned s = cnt[g] / TPK_WAVE * TPK_WAVE + lane; s < slots; s += TPK_WAVE)
            {
                const bool found = s < cnt[g];
                const int2 hit = wave_hits[g * BT_HIT_STRIDE + lane];
                idx4[g * slots + s] = found ? hit.x : -1;
                dist4[g * slots + s] = found ? __int_as_float(hit.y) : -1.0f;
            }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// SORTED: the nsample (<= 64) NEAREST points with squared distance < radius2, nearest first (equal distances: lower row first), instead
// of the first nsample in row order with squared distance <= radius2.  Nothing ends a scan early then: a query that cannot walk takes
// its cloud's rows themselves as candidates.
// unbounded: the radius has no finite square, and accepts points of any cell.
template <bool SORTED>
__global__ void __launch_bounds__(BT_THREADS, SORTED ? 7 : 8) // (wavefronts per SIMD; eight would spill the wider keys)
    bt_query_kernel(int64_t size_y, CellScale scale, float radius2, bool unbounded, int nsample, uint32_t part_mask, const float* __restrict__ x,
                    const float* __restrict__ y, const int64_t* __restrict__ batch_y, const int2* __restrict__ cloud_rows,
                    const float4* __restrict__ records, const int* __restrict__ table, const int* __restrict__ chunk_ends,
                    int64_t* __restrict__ idx, float* __restrict__ dist)
{
    constexpr int WAVES = BT_THREADS / TPK_WAVE;
    __shared__ int2 hits[WAVES][BT_QUERIES * BT_HIT_STRIDE]; // (row, bits of the squared distance)
    __shared__ int marks[WAVES][TPK_WAVE];

    const int lane = threadIdx.x & (TPK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TPK_WAVE);
    const int64_t q0 = (static_cast<int64_t>(blockIdx.x) * WAVES + wave) * BT_QUERIES;
    if (q0 >= size_y)
        return; // (no workgroup barrier anywhere in this kernel)
    const int group = lane / BT_GROUP, sub = lane % BT_GROUP, group_lane = group * BT_GROUP;
    const bool real = q0 + group < size_y;
    const int64_t q = real ? q0 + group : q0;
    int2* const my_hits = hits[wave] + group * BT_HIT_STRIDE;
    int* const my_marks = marks[wave];
    TPK_WORK_DECL

    const float qx = y[q * 3 + 0], qy = y[q * 3 + 1], qz = y[q * 3 + 2];
    const int2 cloud = cloud_rows[q];
    const int s0 = cloud.x, s1 = real ? cloud.y : cloud.x;

    // The runs of buckets that the cube around the ball touches, one per lane.
    const float lx = (qx - scale.reach) * scale.inverse_x, hx = (qx + scale.reach) * scale.inverse_x;
    const float ly = (qy - scale.reach) * scale.inverse_yz, hy = (qy + scale.reach) * scale.inverse_yz;
    const float lz = (qz - scale.reach) * scale.inverse_yz, hz = (qz + scale.reach) * scale.inverse_yz;
    int x0, y0, z0, nx, ny, nz;
    // (cells so far out that a float has no fraction left are seldom)
    const float farthest = fmaxf(fmaxf(fmaxf(-lx, hx), fmaxf(-ly, hy)), fmaxf(-lz, hz));
    if (__ballot(!(farthest < BT_FAR && qx == qx && qy == qy && qz == qz)) == 0)
    {
        x0 = static_cast<int>(floorf(lx)), nx = static_cast<int>(floorf(hx)) - x0 + 1;
        y0 = static_cast<int>(floorf(ly)), ny = static_cast<int>(floorf(hy)) - y0 + 1;
        z0 = static_cast<int>(floorf(lz)), nz = static_cast<int>(floorf(hz)) - z0 + 1;
    }
    else
    {
        x0 = bt_scaled_cell(lx), nx = bt_scaled_cell(hx) - x0 + 1;
        y0 = bt_scaled_cell(ly), ny = bt_scaled_cell(hy) - y0 + 1;
        z0 = bt_scaled_cell(lz), nz = bt_scaled_cell(hz) - z0 + 1;
    }
    bool scan = unbounded || !(nx >= 1 && nx <= BT_MOST_X && ny >= 1 && ny <= 3 && nz >= 1 && nz <= 3);
    const int runs = scan ? 0 : ny * nz;
    // (up to eight runs: the upper eight lanes take the second halves of runs that cross from one chunk to the next)
    const int run = runs <= 8 ? sub & 7 : sub;
    const bool second = runs <= 8 && sub >= 8;
    int start = 0, size = 0;
    bool crosses = false;
    if (run < runs && s1 > s0)
    {
        const int iz = (run >= ny ? 1 : 0) + (run >= 2 * ny ? 1 : 0);
        const BtRow row = bt_row(y0 + run - iz * ny, z0 + iz, batch_y[q]);
        const uint32_t first = bt_bucket(row, x0, part_mask), last = bt_bucket(row, x0 + nx - 1, part_mask);
        crosses = first / BT_CHUNK != last / BT_CHUNK;
        if (!second || crosses)
        {
            const uint32_t from = second ? last & ~static_cast<uint32_t>(BT_CHUNK - 1) : first;
            const uint32_t to = !second && crosses ? first | (BT_CHUNK - 1) : last;
            start = table[from];
            size = ((to + 1) % BT_CHUNK == 0 ? chunk_ends[to / BT_CHUNK] : table[to + 1]) - start;
        }
    }
    if (runs > 8)
        scan = ((__ballot(crosses) >> group_lane) & 0xffff) != 0;
    const int before = row_exclusive_sum(size);
    int total = row_last(before + size, lane);
    scan = scan || total > s1 - s0;
    if (scan)
        total = SORTED ? s1 - s0 : 0;

    int cnt = 0;             // hits kept so far, the same in all lanes of a query
    // Once nsample hits are kept, a candidate has to come before the last of them: in the order of rows s0 .. s0 + wanted, or
    // (SORTED) with a smaller distance than `limit`, or that distance and a row below `limit_row`.
    unsigned wanted = s1 - s0;
    float limit = radius2;
    int limit_row = 0;
    const unsigned group_low = group < 2 ? 0xffffu << group_lane : 0, group_high = group < 2 ? 0 : 0xffffu << (group_lane - 32);
    int most_total = rows_max(total);
    auto record_at = [&](int at) __attribute__((always_inline)) {
        return records[static_cast<uint32_t>(at)];
    };
    const bool any_rows = SORTED && __ballot(scan && s1 > s0) != 0;
    const int origin = start - before; // candidate c of a query lies at origin + c, for the c of this lane's run
    // Four runs at most, in the lanes 0 .. 3 of the query, nearly always: where they begin and lie, known to all its lanes.
    const bool few = __ballot(crosses || runs > 4) == 0;
    const int second_at = row_lane<1>(before), third_at = row_lane<2>(before), fourth_at = row_lane<3>(before);
    const int o0 = row_lane<0>(origin), o1 = row_lane<1>(origin), o2 = row_lane<2>(origin), o3 = row_lane<3>(origin);
    auto of_few = [&](int c) __attribute__((always_inline)) { return c + (c < third_at ? (c < second_at ? o0 : o1) : (c < fourth_at ? o2 : o3)); };
    if constexpr (!SORTED)
    {
        // A run of cells holds 5 to 13 times what the ball itself does, on a surface and in space, but a query beside a surface whose
        // cells it touches may have a hundredth.  Where the scan would be sooner with half of the candidates in the ball, but not with a
        // sixty-fourth, a few of them at equal distances tell.  (100000 points in a room of 8, 12500 queries: always an eighth, radius 0.6,
        // 177 us instead of 133; asked from 1024 candidates on, 24000 points of twelve rooms, radius 2, 63 instead of 35; asked whatever
        // they say, radius 4, 26 instead of 23.)
        const float rows = static_cast<float>(s1 - s0), slots = static_cast<float>(nsample), candidates = static_cast<float>(total);
        auto scan_is_sooner = [&](float share, float more) __attribute__((always_inline)) {
            return scan_is_shorter(rows, slots, candidates * share, more, BT_SCAN_STEP);
        };
        const bool may = total > BT_LONG && scan_is_sooner(BT_MOST_HIT, candidates);
        scan = scan || (may && scan_is_sooner(BT_LEAST_HIT, candidates));
        const bool asks = may && !scan;
        total = scan ? 0 : total;
        if (__ballot(asks) != 0)
        {
            int in = 0;
            if (few)
            {
                float4 p[BT_SAMPLES];
                const int apart = total / (BT_SAMPLES * BT_GROUP);
#pragma unroll
                for (int j = 0; j < BT_SAMPLES; ++j)
                    p[j] = record_at(asks ? of_few(apart * (j * BT_GROUP + sub)) : 0);
#pragma unroll
                for (int j = 0; j < BT_SAMPLES; ++j)
                {
                    const unsigned long long all = __ballot(tpk_dist2(qx, qy, qz, p[j].x, p[j].y, p[j].z) <= radius2);
                    TPK_WORK_ADD(asks ? 1 : 0);
                    in += __builtin_popcount(static_cast<unsigned>(all) & group_low) + __builtin_popcount(static_cast<unsigned>(all >> 32) & group_high);
                }
            }
            const float share = few ? fmaxf(static_cast<float>(in), 0.5f) * (1.0f / (BT_SAMPLES * BT_GROUP)) : 0.125f;
            scan = scan || (asks && scan_is_sooner(share, candidates));
            total = scan ? 0 : total;
        }
    }
    int alone = 0; // candidates of a walk that the whole wavefront makes for this query, behind the others' walks
    if constexpr (!SORTED)
    {
        alone = few && nsample <= BT_KEPT && total > BT_ALONE ? total : 0;
        total = alone > 0 ? 0 : total;
    }
    most_total = rows_max(total);
    auto fetch = [&](int c0) __attribute__((always_inline)) {
        const int c = c0 + sub;
        int at = c;
        if (few)
            at = of_few(c);
        else
        {
            // Whose candidate is c?  Every run's lane marks the slot of its first candidate of this step with its own
            // number; a running maximum over the row carries the number on to the run's other candidates.  (What a lane reads
            // back was written by other lanes: fences for the compiler, no instructions.)
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            my_marks[lane] = 0;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if (size > 0 && before < c0 + BT_GROUP && before + size > c0)
                my_marks[group_lane + max(before - c0, 0)] = sub;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            at += __builtin_amdgcn_ds_bpermute((group_lane + row_inclusive_max(my_marks[lane])) * 4, origin);
        }
        if (any_rows && scan)
        {
            const int64_t row = s0 + min(c, total - 1);
            return c < total ? make_float4(x[row * 3 + 0], x[row * 3 + 1], x[row * 3 + 2], __int_as_float(static_cast<int>(row))) : record_at(0);
        }
        return record_at(c < total ? at : 0);
    };
    int c0 = 0;
    for (;;)
    {
        for (bool full = false; c0 < most_total && !full;)
        {
            float4 p[BT_AHEAD];
#pragma unroll
            for (int j = 0; j < BT_AHEAD; ++j)
                if (j == 0 || c0 + j * BT_GROUP < most_total)
                    p[j] = fetch(c0 + j * BT_GROUP);
#pragma unroll
            for (int j = 0; j < BT_AHEAD; ++j)
            {
                if (c0 >= most_total || full)
                    break;
                const bool has = c0 + sub < total;
                const float d = tpk_dist2(qx, qy, qz, p[j].x, p[j].y, p[j].z);
                TPK_WORK_ADD(has ? 1 : 0);
                const int row = __float_as_int(p[j].w);
                const bool near_enough = SORTED ? d < limit || (d == limit && row < limit_row) : d <= radius2;
                const bool hit = has && near_enough && static_cast<unsigned>(row - s0) < wanted;
                const unsigned long long all = __ballot(hit);
                c0 += BT_GROUP;
                if (all == 0)
                    continue;
                const unsigned low = static_cast<unsigned>(all) & group_low, high = static_cast<unsigned>(all >> 32) & group_high;
                const unsigned slot = __builtin_amdgcn_mbcnt_hi(high, __builtin_amdgcn_mbcnt_lo(low, cnt));
                if (hit)
                    my_hits[slot] = make_int2(row, __float_as_int(d));
                cnt += __builtin_popcount(low) + __builtin_popcount(high);
                full = __ballot(cnt > BT_HITS) != 0;
            }
        }
        // Full: the nsample lowest rows are kept and the walk goes on, or the query is scanned for.  (Once rows are kept
        // their number says nothing about the ball any more.)
        const bool full = cnt > BT_HITS;
        if (!SORTED && full && wanted == static_cast<unsigned>(s1 - s0))
        {
            const float tested = static_cast<float>(min(c0, total)), left = static_cast<float>(total) - tested;
            const float ball = static_cast<float>(cnt) * static_cast<float>(total) * __builtin_amdgcn_rcpf(tested);
            scan = nsample > BT_KEPT || scan_is_shorter(static_cast<float>(s1 - s0), static_cast<float>(nsample), ball, left, BT_SCAN_STEP_LATER);
            total = scan ? 0 : total;
            cnt = scan ? 0 : cnt;
        }
        most_total = rows_max(total);
        const bool ends = c0 >= most_total, ordered = ends || cnt > BT_HITS;
        order_hits<SORTED>(hits[wave], ordered ? cnt : 0, lane, nsample);
        if (ordered && cnt >= nsample)
        {
            cnt = nsample;
            const int2 last = my_hits[nsample - 1];
            if constexpr (SORTED)
            {
                limit = __int_as_float(last.y);
                limit_row = last.x;
            }
            else
                wanted = last.x - s0;
        }
        if (ends)
            break;
    }

    // The hits in order, then the padding.
    int64_t* const idx4 = idx + q0 * nsample;
    float* const dist4 = dist + q0 * nsample;
    if (real && (SORTED || (!scan && alone == 0)))
        for (int s = sub; s < nsample; s += BT_GROUP)
        {
            const bool found = s < cnt;
            const int2 hit = my_hits[found ? s : 0];
            const uint32_t out = static_cast<uint32_t>(group * nsample + s);
            idx4[out] = found ? hit.x : -1;
            dist4[out] = found ? __int_as_float(hit.y) : -1.0f;
        }

    // The queries with long lists of candidates, one after the other: sixteen lanes take a wavefront as many steps as its longest query, and
    // on a chip that few queries do not fill nothing hides the others' idle lanes (17000 queries of 200000 points in a room of 8, radius 1: 118 / 314 us
    // -> 87 / 225).  (In front of the others' walks, whose registers they then crowd: 300000 queries, radius 0.1, 82 / 97 -> 101 / 129.)
    if constexpr (!SORTED)
    {
        unsigned long long longer = __ballot(sub == 0 && alone > 0);
        while (longer != 0)
        {
            const int from = __builtin_ctzll(longer); // the query's first lane
            longer &= longer - 1;
            const bool mine = from == group_lane;
            const int its_total = tpk_read_lane(alone, from), b1 = tpk_read_lane(second_at, from), b2 = tpk_read_lane(third_at, from),
                      b3 = tpk_read_lane(fourth_at, from), i0 = tpk_read_lane(o0, from), i1 = tpk_read_lane(o1, from), i2 = tpk_read_lane(o2, from),
                      i3 = tpk_read_lane(o3, from), first = tpk_read_lane(s0, from), rows = tpk_read_lane(s1, from) - first;
            const float x1 = to_vector_register(tpk_read_lane(qx, from)), y1 = to_vector_register(tpk_read_lane(qy, from)),
                        z1 = to_vector_register(tpk_read_lane(qz, from));
            int2* const list = hits[wave] + from / BT_GROUP * BT_HIT_STRIDE;
            int its_cnt = 0, c0 = 0;
            unsigned its_wanted = rows;
            bool gives_up = false;
            for (;;)
            {
                while (c0 < its_total && its_cnt <= BT_ALONE_HITS)
                {
                    float4 p[BT_ALONE_AHEAD];
#pragma unroll
                    for (int j = 0; j < BT_ALONE_AHEAD; ++j)
                        if (j == 0 || c0 + j * TPK_WAVE < its_total)
                        {
                            const int c = c0 + j * TPK_WAVE + lane;
                            p[j] = record_at(c < its_total ? c + (c < b2 ? (c < b1 ? i0 : i1) : (c < b3 ? i2 : i3)) : 0);
                        }
#pragma unroll
                    for (int j = 0; j < BT_ALONE_AHEAD; ++j)
                    {
                        if (c0 >= its_total || its_cnt > BT_ALONE_HITS)
                            break;
                        const bool has = c0 + lane < its_total;
                        const float d = tpk_dist2(x1, y1, z1, p[j].x, p[j].y, p[j].z);
                        TPK_WORK_ADD(has ? 1 : 0);
                        const int row = __float_as_int(p[j].w);
                        const bool hit = has && d <= radius2 && static_cast<unsigned>(row - first) < its_wanted;
                        const unsigned long long all = __ballot(hit);
                        c0 += TPK_WAVE;
                        if (all == 0)
                            continue;
                        if (hit)
                            list[__builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(all >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(all), its_cnt))] =
                                make_int2(row, __float_as_int(d));
                        its_cnt += __builtin_popcountll(all);
                    }
                }
                const bool ends = c0 >= its_total;
                if (!ends && its_wanted == static_cast<unsigned>(rows))
                {
                    const float tested = static_cast<float>(c0);
                    gives_up = scan_is_shorter(static_cast<float>(rows), static_cast<float>(nsample),
                                               static_cast<float>(its_cnt) * static_cast<float>(its_total) * __builtin_amdgcn_rcpf(tested),
                                               static_cast<float>(its_total) - tested, BT_SCAN_STEP_LATER);
                    if (gives_up)
                        break;
                }
                order_hits<false>(hits[wave], mine ? its_cnt : 0, lane, nsample);
                if (its_cnt >= nsample)
                {
                    its_cnt = nsample;
                    its_wanted = __builtin_amdgcn_readfirstlane(list[nsample - 1].x) - first;
                }
                if (ends)
                    break;
            }
            scan = scan || (mine && gives_up);
            if (!gives_up && lane < nsample)
            {
                const bool found = lane < its_cnt;
                const int2 hit = list[lane];
                const uint32_t out = static_cast<uint32_t>(from / BT_GROUP * nsample + lane);
                idx4[out] = found ? hit.x : -1;
                dist4[out] = found ? __int_as_float(hit.y) : -1.0f;
            }
        }
    }

    // The queries that were given up, those of one cloud together.
    unsigned long long left = __ballot(!SORTED && real && scan && sub == 0);
    while (left != 0)
    {
        const int from = __builtin_ctzll(left);
        const int first = tpk_read_lane(s0, from), end = tpk_read_lane(s1, from);
        const unsigned long long with = left & __ballot(s0 == first && s1 == end);
        left &= ~with;
        bt_scan_rows(x, first, end, with, qx, qy, qz, radius2, nsample, lane, hits[wave], idx4, dist4 TPK_WORK_ARG);
    }
    TPK_WORK_FLUSH
}

struct TableLayout
{
    int64_t buckets;
    size_t records, table, chunk_ends, ranks, cloud_rows, placed, total;
};

TableLayout table_layout(int64_t size_x, int64_t size_y)
{
    auto up = [](size_t v) { return (v + 255) & ~static_cast<size_t>(255); };
    TableLayout l;
    l.buckets = 2 * BT_CHUNK * BT_PARTS; // (a run that wraps around its part ends in another chunk than it starts in)
    while (l.buckets < 2 * size_x)
        l.buckets *= 2;
    size_t pos = 0;
    l.records = pos;
    pos = up(pos + static_cast<size_t>(size_x) * sizeof(float4));
    l.table = pos;
    pos = up(pos + static_cast<size_t>(l.buckets) * sizeof(int));
    l.chunk_ends = pos;
    pos = up(pos + static_cast<size_t>(l.buckets / BT_CHUNK) * sizeof(int));
    l.ranks = pos;
    pos = up(pos + static_cast<size_t>(size_x) * sizeof(int));
    l.cloud_rows = pos;
    pos = up(pos + static_cast<size_t>(size_y) * sizeof(int2));
    l.placed = pos;
    pos = up(pos + sizeof(int));
    l.total = pos;
    return l;
}

// Five launches and an atomic per support point have to pay: with fewer queries, or with fewer than a twelfth as many as points, the walk
// over bins (two launches) answers a call in row order as soon or sooner.  33000 points, 4100 queries 20.7 us over bins, 23 here,
// 33000 queries 32 and 24; 100000 points, 12500 queries 32 and 26; 212000 points, 13250 queries 33 and 35, 26600 queries 38 and 37.
// Sorted neighbours cost the walk over bins more (a list of 64 keys, merged at every step with a hit), so it is the sooner one only for
// few queries of a large array.  Over bins and here, us, radius 0.1 / 0.3 / 1.5 with 16 / 64 / 16 slots in rooms of 8:
//     20000 points, 16 queries   23 / 22 / 81 and 19 / 24 / 55;  50000 points, 512 queries  24 / 26 / 123 and 21 / 27 / 109
//     100000 points, 512 queries  25 / 31 / 157 and 24 / 34 / 186, 2048 queries  26 / 33 / 168 and 24 / 35 / 181
//     200000 points, 2048 queries  31 / 50 / 223 and 33 / 47 / 319, 8192 queries  37 / 57 / 466 and 34 / 49 / 326
//     400000 points, 512 queries  37 / 60 / 314 and 52 / 75 / 660, 8192 queries  51 / 88 / 656 and 53 / 84 / 626
//     a million points, 16 queries  42 / 70 / 633 and 100 / 147 / 1557, 12500 queries  95 / 192 / 1771 and 103 / 198 / 2408
// (In between, where a ball touches many bins of every window, the walk over bins is the slower one at every number of queries: a million points,
// radius 0.6, 512 queries 630 and 347.  The host does not know the clouds' extent.)
constexpr int64_t BT_MIN_QUERIES = 8192, BT_MOST_SHARE = 12, BT_SORTED_SHARE = 64, BT_SORTED_POINTS = 65536;

bool table_supported(int64_t size_x, int64_t size_y, int nsample)
{
    // Small problems are served as fast by the all-pairs scan; rows and buckets are 32-bit here.
    return size_x >= 8192 && size_y > 0 && nsample > 0 && size_x < (1LL << 30);
}

} // namespace

size_t tpk_table_ball_query_workspace_bytes(int64_t size_x, int64_t size_y, int nsample)
{
    return table_supported(size_x, size_y, nsample) ? table_layout(size_x, size_y).total : 0;
}

bool tpk_table_ball_query_pays(int64_t size_x, int64_t size_y, bool sorted)
{
    return sorted ? size_x < BT_SORTED_POINTS || size_y >= size_x / BT_SORTED_SHARE : size_y >= BT_MIN_QUERIES && size_y >= tpk_ceil_div(size_x, BT_MOST_SHARE);
}

int tpk_table_ball_query_partial(int64_t size_x, int64_t size_y, float radius, float radius2, int nsample, bool sorted, const float* x,
                                 const float* y, const int64_t* batch_x, const int64_t* batch_y, int64_t* idx, float* dist, void* workspace,
                                 size_t workspace_bytes, hipStream_t s)
{
    if (!table_supported(size_x, size_y, nsample) || !tpk_table_ball_query_pays(size_x, size_y, sorted) || (sorted && nsample > TPK_WAVE))
        return TPK_ERR_UNSUPPORTED;
    const TableLayout l = table_layout(size_x, size_y);
    if (!workspace || workspace_bytes < l.total)
        return TPK_ERR_UNSUPPORTED; // (the bin walk makes do with less)
    if (reinterpret_cast<uintptr_t>(workspace) & 255u)
        return TPK_ERR_WORKSPACE;
    char* w = static_cast<char*>(workspace);
    float4* records = reinterpret_cast<float4*>(w + l.records);
    int* table = reinterpret_cast<int*>(w + l.table);
    int* chunk_ends = reinterpret_cast<int*>(w + l.chunk_ends);
    int* ranks = reinterpret_cast<int*>(w + l.ranks);
    int* placed = reinterpret_cast<int*>(w + l.placed);
    const CloudRows rows{batch_x, batch_y, static_cast<int>(size_x), size_y, reinterpret_cast<int2*>(w + l.cloud_rows)};
    CellScale scale;
    scale.reach = bt_reach(radius);
    scale.inverse_x = 1.0f / (BT_WIDTH_X * scale.reach);
    scale.inverse_yz = 1.0f / (BT_WIDTH_YZ * scale.reach);
    const uint32_t part_mask = static_cast<uint32_t>(l.buckets / BT_PARTS - 1);
    const int n = static_cast<int>(size_x);

    const int64_t point_blocks = tpk_ceil_div(size_x, BT_THREADS);
    const int count_threads = size_x < BT_COUNT_MEDIUM ? BT_COUNT_THREADS / 4 : size_x < BT_COUNT_LARGE ? BT_COUNT_THREADS / 2 : BT_COUNT_THREADS;
    const int64_t count_blocks = tpk_ceil_div(size_x, count_threads), row_blocks = tpk_ceil_div(size_y, count_threads);
    const int64_t query_blocks = tpk_ceil_div(size_y, BT_THREADS / BT_GROUP);
    if (query_blocks > 0x7fffffffLL || count_blocks + row_blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(bt_clear_kernel, dim3(static_cast<unsigned>(tpk_ceil_div(l.buckets / 4, BT_THREADS))), dim3(BT_THREADS), 0, s,
                       l.buckets / 4, reinterpret_cast<int4*>(table));
    auto* const count_kernel = size_x < BT_COUNT_MEDIUM  ? &bt_count_kernel<BT_COUNT_THREADS / 4>
                               : size_x < BT_COUNT_LARGE ? &bt_count_kernel<BT_COUNT_THREADS / 2>
                                                         : &bt_count_kernel<BT_COUNT_THREADS>;
    hipLaunchKernelGGL(count_kernel, dim3(static_cast<unsigned>(count_blocks + row_blocks)), dim3(count_threads), 0, s, n,
                       static_cast<unsigned>(count_blocks), x, batch_x, scale, part_mask, table, ranks, placed, rows);
    hipLaunchKernelGGL(bt_places_kernel, dim3(static_cast<unsigned>(l.buckets / BT_CHUNK)), dim3(BT_SCAN_THREADS), 0, s,
                       reinterpret_cast<int4*>(table), chunk_ends, placed);
    hipLaunchKernelGGL(bt_records_kernel, dim3(static_cast<unsigned>(point_blocks)), dim3(BT_THREADS), 0, s, n, x, batch_x, scale, part_mask,
                       table, ranks, records);
    const bool unbounded = !(radius2 < INFINITY);
    if (sorted)
        hipLaunchKernelGGL((bt_query_kernel<true>), dim3(static_cast<unsigned>(query_blocks)), dim3(BT_THREADS), 0, s, size_y, scale, radius2, unbounded,
                           nsample, part_mask, x, y, batch_y, rows.rows, records, table, chunk_ends, idx, dist);
    else
        hipLaunchKernelGGL((bt_query_kernel<false>), dim3(static_cast<unsigned>(query_blocks)), dim3(BT_THREADS), 0, s, size_y, scale, radius2, unbounded,
                           nsample, part_mask, x, y, batch_y, rows.rows, records, table, chunk_ends, idx, dist);
    return tpk_launch_status();
}
