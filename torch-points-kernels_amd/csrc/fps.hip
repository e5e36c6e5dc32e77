// Furthest point sampling: npoint-1 dependent rounds of "update every point's distance to
// the chosen set, pick the point whose distance is largest".
//
// One workgroup (one compute unit) owns a cloud for the whole call; the rounds of a cloud
// depend on each other, so a call runs as many workgroups as there are clouds.  Four kernels
// by cloud size:
//   up to 256 points     fps_wave_kernel: one wavefront, a sample at a time;
//   up to 16384 points   fps_pool_kernel: up to 16 points per lane in registers, cloud ordered along
//                        a space filling curve so that most updates can be skipped exactly; dozens of
//                        samples per round from a pool (described at the kernel);
//   up to 163840 points  fps_cells_batched_kernel: the cloud ordered along the curve into cells of 64
//                        points that stay in memory (the caller's workspace); boxes, largest
//                        distance and best point of every cell in LDS; a round touches only
//                        the cells the new sample can change (described at the kernel);
//   larger clouds        fps_streaming_kernel: every point updated every round, points streamed from
//                        global memory, running minima in a workspace provided by the caller.
// In all of them the chosen point's coordinates travel through LDS with the selection: the
// chosen point is never re-read from memory.
//
// Semantics follow the reference kernel (cuda/src/sampling_gpu.cu:17-144): start at point
// 0; squared distances; points whose squared norm is <= 1e-3 are neither updated nor
// eligible; if no point is eligible the pick is 0.  Equal maxima resolve as its block
// reduction does: with BS = the reference's block size (largest power of two <= n, at
// most 512; cuda/include/cuda_utils.h:13-18), reference thread (k mod BS) keeps the lowest
// k among its own equal maxima, and the halving tree then prefers the thread whose number
// has the smaller bit-reversal.  Both rules together are "smallest tie key", with
//   key(k) = bitrev(k mod BS) * ceil(n / BS) + floor(k / BS).
#include "coarse_order.h"

#include <cmath>
#include <type_traits>

namespace {

constexpr int FPS_THREADS = 1024;
constexpr int FPS_WAVES = FPS_THREADS / TPK_WAVE;
constexpr int FPS_REGISTER_POINTS = 16384; // largest cloud kept in registers

struct WaveRecord
{
    int val;     // bits of the wavefront's largest distance (-1.0f: no eligible point)
    unsigned tk; // tie key of the point holding it
    int k;       // its index in the cloud
    float x, y, z;
};

// Distances are >= 0 and the "nothing eligible" marker is -1.0f, so the bit patterns order
// like signed integers.
__device__ __forceinline__ int ordered_bits(float v)
{
    return __float_as_int(v);
}

// Lane of the wavefront holding the largest `val`; among equals the smallest tie key.
__device__ __forceinline__ int winning_lane(int val, unsigned tk, int& wave_val)
{
    wave_val = wave_max_i32(val);
    const unsigned long long top = __ballot(val == wave_val);
    if (__builtin_popcountll(top) == 1)
        return __builtin_ctzll(top);
    const unsigned cand = val == wave_val ? tk : 0xFFFFFFFFu;
    const unsigned lowest = wave_min_u32(cand);
    return __builtin_ctzll(__ballot(cand == lowest));
}

// Step 3: every wavefront reduces the 16 published records; returns the chosen point.
template <int WAVES>
__device__ __forceinline__ void reduce_records(const WaveRecord* __restrict__ rec, int lane,
                                               float p0x, float p0y, float p0z, int& k,
                                               float& sx, float& sy, float& sz, int& gv_out)
{
    const WaveRecord e = rec[lane & (WAVES - 1)];
    const int gv = __builtin_amdgcn_readfirstlane(row_all_max_i32(e.val));
    gv_out = gv;
    constexpr unsigned wave_bits = (1u << WAVES) - 1u;
    const unsigned top = static_cast<unsigned>(__ballot(e.val == gv)) & wave_bits;
    int w;
    if (__builtin_popcount(top) == 1)
    {
        w = __builtin_ctz(top);
    }
    else
    {
        const unsigned cand = e.val == gv ? e.tk : 0xFFFFFFFFu;
        const unsigned lowest = __builtin_amdgcn_readfirstlane(row_all_min_u32(cand));
        w = __builtin_ctz(static_cast<unsigned>(__ballot(cand == lowest)) & wave_bits);
    }
    k = __builtin_amdgcn_readlane(e.k, w);
    sx = tpk_read_lane(e.x, w);
    sy = tpk_read_lane(e.y, w);
    sz = tpk_read_lane(e.z, w);
    if (gv < 0)
    {
        // No eligible point in the whole cloud: the reference's reduction yields index 0.
        k = 0;
        sx = p0x;
        sy = p0y;
        sz = p0z;
    }
}

// A point takes part unless its squared norm is <= 1e-3 (compared in double precision, as
// the reference's literal makes it).
__device__ __forceinline__ bool eligible(float x, float y, float z)
{
    const float mag = (x * x) + (y * y) + (z * z);
    return !(static_cast<double>(mag) <= 1e-3);
}

// ---------------------------------------------------------------------------------------
// Register-resident kernel with exact pruning and pools of samples, for clouds of 257 to 16384 points.
//
// Pools.  A round takes many samples.  Let the pool be all points whose running minimum lies above some
// floor; no point outside it holds more than the floor, and minima only fall.  So as long as the largest
// minimum inside the pool lies above the floor, it is the largest of the cloud and its point the next sample.
// What the pool's points do to each other decides the whole sequence at once: in the order of their minima
// (equal ones by the tie key) a point is taken unless one taken before it is closer to it than its minimum.
// Every wavefront forms the distances of its share of the pool's pairs and leaves, per point, a mask of who would
// lower it; then all points whose lowering points are decided are decided together, two or three passes of a dozen
// scalar instructions.  A point lowered by those taken, but not to the floor, would have its turn again: the round
// is cut where the largest of these stands, and what lies below waits for the next pool.  A pool of 54 gives about 38
// samples.  (The version before let one wavefront take sample after sample, a chain of 40 dependent instructions
// each, while the others updated: 31 samples per round, 0.1 us each.)
//
// A round is: gather the pool in LDS; barrier; (if it holds more than 64, one wavefront picks the best 64; barrier;)
// the pairs; barrier; decide, in every wavefront alike; update this wavefront's points with all samples.  What
// share below the largest minimum makes a pool of the wanted size is carried from round to round.  At 16384 points a round
// takes 13000 clocks: updates 5000, gathering 2200, waiting for the busiest wavefront 2000, the pool 4000.
// 16 clouds of 16384 points, 4096 samples: 853 -> 602 us (uneven clouds 938 -> 725); 4096 points 235 -> 158, 1024 85 -> 63.
//
// Pruning.  A point's running minimum changes only if its distance to the new sample is smaller
// than that minimum, and no minimum exceeds the one the sample held.  So a set of
// points whose bounding box is further from the sample than the square root of that value cannot
// change, and its update can be skipped without changing any result.  To make such sets exist, the
// kernel first orders the cloud along a Hilbert curve (12-bit position of its cell in a 16^3 grid,
// counting sort in LDS) and cuts the curve into cells of 64 * GS consecutive points.  A cell is GS
// registers of the 64 lanes of one wavefront; cells go round-robin to the wavefronts, so the cells around a
// sample belong to different ones.  A wavefront tests its boxes against all samples of a round, a lane each, and updates
// only what is reached.  The fp32 box distance is compared with a relative margin of 3e-6, several times the rounding error
// of either side, so a skipped update is provably a no-op.  (Cells of 64, 128, 256 points: 749 / 612 / 603 us on even clouds,
// 806 / 736 / 720 on uneven ones at 16384 points, 181 / 169 / 174 and 193 / 186 / 213 at 4096.)
//
// One sample per round.  The first samples drop so many minima that a pool gives one to four of them; and when more
// points hold the same value than a pool takes, when nothing above zero is left, or when a coordinate is not finite
// (such a point never falls to zero), a pool gives none.  Then every wavefront offers its best point, one barrier, and all
// find the best of those: 4900 clocks a sample at 16384 points, most of them for the rank among equal minima that all
// wavefronts look for in turn.  1024 of 16384 points on 1728 places, nearly all of them taken this way: 2300 us.
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ unsigned tie_key(int k, int log2_bs, int ref_groups)
{
    const unsigned bs_mask = (1u << log2_bs) - 1u;
    const unsigned rev = log2_bs ? (__brev(static_cast<unsigned>(k) & bs_mask) >> (32 - log2_bs)) : 0u;
    return rev * static_cast<unsigned>(ref_groups) + (static_cast<unsigned>(k) >> log2_bs);
}

// LDS atomics without return value, issued as written: one instruction for the active lanes
// (the compiler would otherwise wrap a same-address atomic in a loop over those lanes).
__device__ __forceinline__ unsigned lds_offset(const void* p)
{
    return static_cast<unsigned>(reinterpret_cast<unsigned long long>(
        (const __attribute__((address_space(3))) char*)p));
}
__device__ __forceinline__ void lds_or_u32(unsigned* p, unsigned v)
{
    asm volatile("ds_or_b32 %0, %1" ::"v"(lds_offset(p)), "v"(v) : "memory");
}

// Largest value of the wavefront as a scalar: DPP maxima inside the rows of 16 lanes, then from row to row; six
// dependent steps and one lane read.
__device__ __forceinline__ int wave_max_to_scalar(int v)
{
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true));  // quad_perm [1,0,3,2]
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true));  // quad_perm [2,3,0,1]
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, true)); // row_half_mirror
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x140, 0xF, 0xF, true)); // row_mirror
    v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, 0x142, 0xA, 0xF, false)); // row_bcast:15 into rows 1 and 3
    v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, 0x143, 0xC, 0xF, false)); // row_bcast:31 into rows 2 and 3
    return __builtin_amdgcn_readlane(v, TPK_WAVE - 1);
}

// `v`, of which the compiler shall not know that it stays the same: what is computed from it is computed where it is used
// instead of once before the loop and kept in registers that the points need.
__device__ __forceinline__ int not_hoisted(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// Calls f with the slot (LOW .. LOW + N - 1, the same in all lanes) as a constant: log2(N) branches instead of N in a row,
// each of them 24 clocks of all wavefronts of a SIMD (1024 of 16384 points on 1728 places, taken one by one: 2590 -> 2297 us).
template <int LOW, int N, typename F>
__device__ __forceinline__ void with_slot(int slot, F&& f)
{
    if constexpr (N == 1)
        f(std::integral_constant<int, LOW>{});
    else if (slot < LOW + N / 2)
        with_slot<LOW, N / 2>(slot, f);
    else
        with_slot<LOW + N / 2, N / 2>(slot, f);
}

// Position on the sorted curve of member `e` of group `g` held by lane `lane` of wavefront `wave`.
template <int WAVES, int GS>
__device__ __forceinline__ int sorted_position(int g, int wave, int e, int lane)
{
    return ((g * WAVES + wave) * GS + e) * TPK_WAVE + lane;
}

constexpr int POOL_CAPACITY = 4 * TPK_WAVE; // points gathered at most; the best 64 are sampled
constexpr int POOL_TARGET = 64;             // (56, 64, 72, 84: 611 / 603 / 601 / 606 us at 16384 points)
constexpr int POOL_TRIES = 12;

// ORDERED: the cloud is ordered along the curve and updates are pruned.  Small clouds are taken as they come.
template <int PPT, int WAVES, int GS, bool ORDERED>
__global__ __launch_bounds__(WAVES* TPK_WAVE) void fps_pool_kernel(
    int n, int npoint, int log2_bs, int ref_groups, int key_capacity,
    const float* __restrict__ xyz, int32_t* __restrict__ out)
{
    constexpr int THREADS = WAVES * TPK_WAVE;
    constexpr int NG = PPT / GS;
    // samples taken one by one before the first pool (1, 8, 16, 32: 74 / 72 / 69 / 71 us for 256 of 1024 points, 625 / 610 / 606 /
    // 611 for 4096 of 16384; 2048 points 102 / 98 / 102 / 106)
    constexpr int OPENING = ORDERED && PPT <= 2 ? 8 : 16;
    constexpr int ROWS = TPK_WAVE / WAVES; // rows of the pool's relation that a wavefront works out
    static_assert(PPT <= 16 && NG * GS == PPT && ROWS * WAVES == TPK_WAVE && ROWS % 4 == 0, "whole groups, whole rows");
    // key_capacity keys (curve position << 20) | index in curve order, kept for the whole kernel; then, during
    // set-up, key_capacity unsorted keys and the bins of the counting sort
    extern __shared__ __align__(16) unsigned sort_keys[];
    unsigned* const unsorted = sort_keys + key_capacity;
    int* const bins = reinterpret_cast<int*>(unsorted + key_capacity); // CURVE_BINS words
    __shared__ int wave_totals[WAVES];
    __shared__ int cloud_box[6];      // ordered ints: min x,y,z then max x,y,z
    __shared__ __align__(16) float4 group_lo[WAVES * NG], group_hi[WAVES * NG]; // box of every (wavefront, group) cell
    // The pool's points (x, y, z, running minimum) and their places on the curve, rounds in turn: where the ordering had
    // its unsorted keys
    __shared__ __align__(16) float4 pool_room[ORDERED ? 1 : 2 * POOL_CAPACITY];
    __shared__ int pool_place_room[ORDERED ? 1 : 2 * POOL_CAPACITY];
    float4* const pools = ORDERED ? reinterpret_cast<float4*>(unsorted) : pool_room;
    int* const pool_places = ORDERED ? reinterpret_cast<int*>(pools + 2 * POOL_CAPACITY) : pool_place_room;
    static_assert(2 * POOL_CAPACITY * (sizeof(float4) + sizeof(int)) <= CURVE_BINS * sizeof(int), "room for the pools");
    __shared__ __align__(16) float4 best[TPK_WAVE];      // the same of its best 64, if it holds more
    __shared__ int best_place[TPK_WAVE];
    __shared__ __align__(8) int2 best_of;                // how many they are, what they lie above
    __shared__ int pool_count[3];                        // one per attempt, in turn
    __shared__ __align__(8) uint2 pool_blockers[TPK_WAVE]; // per pool point: who, taken before it, lowers it
    __shared__ __align__(8) uint2 pool_before[TPK_WAVE];   // per pool point: who comes before it
    __shared__ __align__(8) uint2 pool_keepers[TPK_WAVE];  // per pool point with a bit in keeps[]: who lowers it, but not out of the pool
    __shared__ __align__(8) unsigned keeps[2][2];          // rounds in turn
    __shared__ __align__(16) float4 offers[2][WAVES]; // every wavefront's best point (x, y, z, running minimum), rounds in turn
    __shared__ int offer_places[2][WAVES];            // and its place on the curve
    __shared__ int not_finite;

    xyz += static_cast<int64_t>(blockIdx.x) * n * 3;
    out += static_cast<int64_t>(blockIdx.x) * npoint;
    const int tid = threadIdx.x;
    const int lane = tid & (TPK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / TPK_WAVE);
    auto original_index = [&](int position) { return ORDERED ? static_cast<int>(sort_keys[position] & 0x3FFFu) : position; };

    // ---- set-up 1 and 2: order the cloud along the curve (curve_order.h)
    if (tid < 3)
        pool_count[tid] = 0;
    if (tid < 4)
        keeps[tid / 2][tid % 2] = 0;
    if (tid == 0)
        not_finite = 0;
    if constexpr (ORDERED)
        curve_order<THREADS>(xyz, n, sort_keys, unsorted, bins, cloud_box, wave_totals);
    else
        __syncthreads();

    // ---- set-up 3: this lane's points.  The curve is cut into cells of 64 * GS consecutive
    // points; cell c belongs to wavefront c % WAVES as its group c / WAVES.  Slot i of a lane =
    // group (i / GS), member (i % GS); see sorted_position().
    float x[PPT], y[PPT], z[PPT];
    int t[PPT];
    bool finite = true;
#pragma unroll
    for (int i = 0; i < PPT; ++i)
    {
        const int q = sorted_position<WAVES, GS>(i / GS, wave, i % GS, lane);
        const int k = original_index(q < n ? q : 0);
        x[i] = xyz[k * 3 + 0];
        y[i] = xyz[k * 3 + 1];
        z[i] = xyz[k * 3 + 2];
    }
#pragma unroll
    for (int i = 0; i < PPT; ++i)
    {
        const bool ok = sorted_position<WAVES, GS>(i / GS, wave, i % GS, lane) < n && eligible(x[i], y[i], z[i]);
        finite = finite && (!ok || (x[i] - x[i] == 0.f && y[i] - y[i] == 0.f && z[i] - z[i] == 0.f));
        t[i] = ordered_bits(ok ? 1e10f : -1.0f);
    }
    if (!finite)
        not_finite = 1;
    if constexpr (ORDERED)
    {
        // a cell belongs to this wavefront alone: reduce over its lanes, plain store
#pragma unroll
        for (int gi = 0; gi < NG; ++gi)
        {
            float lo[3] = {__builtin_inff(), __builtin_inff(), __builtin_inff()};
            float hi[3] = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
#pragma unroll
            for (int e = 0; e < GS; ++e)
            {
                const int i = gi * GS + e;
                const bool ok = t[i] >= 0;
                lo[0] = ok ? fminf(lo[0], x[i]) : lo[0];
                lo[1] = ok ? fminf(lo[1], y[i]) : lo[1];
                lo[2] = ok ? fminf(lo[2], z[i]) : lo[2];
                hi[0] = ok ? fmaxf(hi[0], x[i]) : hi[0];
                hi[1] = ok ? fmaxf(hi[1], y[i]) : hi[1];
                hi[2] = ok ? fmaxf(hi[2], z[i]) : hi[2];
            }
#pragma unroll
            for (int a = 0; a < 3; ++a)
            {
                lo[a] = ordered_int_to_float(wave_min_i32(float_to_ordered_int(lo[a])));
                hi[a] = ordered_int_to_float(wave_max_i32(float_to_ordered_int(hi[a])));
            }
            // a cell without points that take part: a box at infinity, which nothing reaches
            if (lane == 0)
            {
                const bool none = !(lo[0] <= hi[0]);
                group_lo[wave * NG + gi] = none ? make_float4(__builtin_inff(), __builtin_inff(), __builtin_inff(), 0.f) : make_float4(lo[0], lo[1], lo[2], 0.f);
                group_hi[wave * NG + gi] = none ? make_float4(__builtin_inff(), __builtin_inff(), __builtin_inff(), 0.f) : make_float4(hi[0], hi[1], hi[2], 0.f);
            }
        }
    }
    const float p0x = xyz[0], p0y = xyz[1], p0z = xyz[2];
    if (tid == 0)
        out[0] = 0;
    __syncthreads();
    const bool one_by_one = __builtin_amdgcn_readfirstlane(not_finite) != 0;
    TPK_WORK_DECL

    // The updates of the samples held by the lanes of `mask`, a lane each (and by samples[lane] in LDS); `bound`: no running
    // minimum exceeds it when that sample is taken.  (Bit patterns of non-negative floats throughout.)
    auto update = [&](float px, float py, float pz, int bound, unsigned long long mask, const float4* samples) __attribute__((always_inline)) {
        // (two parts in a million and more above the bound: several times the rounding error of either side)
        const float limit = __int_as_float(bound) * 1.000003f;
        int cells = wave * NG;
        unsigned long long reach[NG]; // who reaches a group
#pragma unroll
        for (int gi = 0; gi < NG; ++gi)
        {
            reach[gi] = mask;
            if constexpr (ORDERED)
            {
                if (gi > 0 && gi % 4 == 0) // (four boxes in registers at a time)
                    asm volatile("" : "+s"(cells) : "s"(reach[gi - 1]));
                const float4 lo = group_lo[cells + gi], hi = group_hi[cells + gi];
                const float dx = px - __builtin_amdgcn_fmed3f(px, lo.x, hi.x);
                const float dy = py - __builtin_amdgcn_fmed3f(py, lo.y, hi.y);
                const float dz = pz - __builtin_amdgcn_fmed3f(pz, lo.z, hi.z);
                const float lb = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
                // (a box at infinity: lb = +inf, never live; NaN compares false -> live)
                reach[gi] = __ballot(!(lb >= limit)) & mask;
            }
        }
        if constexpr (!ORDERED)
        {
            // (two samples at a time; every group is reached by all)
            for (unsigned long long left = mask; left != 0; left &= left - 1)
            {
                const int first = __builtin_ctzll(left);
                left &= left - 1;
                const float4 s = samples[first], r = samples[left != 0 ? __builtin_ctzll(left) : first];
                TPK_WORK_ADD(2 * PPT);
#pragma unroll
                for (int i = 0; i < PPT; ++i)
                    t[i] = min(min(t[i], ordered_bits(tpk_dist2(x[i], y[i], z[i], s.x, s.y, s.z))), ordered_bits(tpk_dist2(x[i], y[i], z[i], r.x, r.y, r.z)));
            }
            return;
        }
#pragma unroll
        for (int gi = 0; gi < NG; ++gi)
            for (unsigned long long left = reach[gi]; left != 0; left &= left - 1)
            {
                float4 s = samples[__builtin_ctzll(left)];
                asm volatile("" : "+v"(s.w));
                TPK_WORK_ADD(GS);
#pragma unroll
                for (int e = 0; e < GS; ++e)
                {
                    const int i = gi * GS + e;
                    t[i] = min(t[i], ordered_bits(tpk_dist2(x[i], y[i], z[i], s.x, s.y, s.z)));
                }
            }
    };
    // The same for one sample: a lane tests each group.
    auto update_one = [&](const float4 s, int bound) __attribute__((always_inline)) {
        unsigned long long reach = ~0ull;
        if constexpr (ORDERED)
        {
            const int cell = wave * NG + (lane < NG ? lane : 0);
            const float4 lo = group_lo[cell], hi = group_hi[cell];
            const float dx = s.x - __builtin_amdgcn_fmed3f(s.x, lo.x, hi.x);
            const float dy = s.y - __builtin_amdgcn_fmed3f(s.y, lo.y, hi.y);
            const float dz = s.z - __builtin_amdgcn_fmed3f(s.z, lo.z, hi.z);
            reach = __ballot(!(__builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz)) >= __int_as_float(bound) * 1.000003f));
        }
#pragma unroll
        for (int gi = 0; gi < NG; ++gi)
            if ((reach >> gi & 1ull) != 0ull)
            {
                TPK_WORK_ADD(GS);
#pragma unroll
                for (int e = 0; e < GS; ++e)
                {
                    const int i = gi * GS + e;
                    t[i] = min(t[i], ordered_bits(tpk_dist2(x[i], y[i], z[i], s.x, s.y, s.z)));
                }
            }
    };
    update_one(make_float4(p0x, p0y, p0z, 0.f), ordered_bits(__builtin_inff()));

    int most_left = 0;       // no running minimum exceeds this
    // the pool takes what lies above this much less than it, in bit patterns: 2^23 is a factor of two
    int gap = 1 << 21;
    int pause = OPENING, penalty = 1; // samples to take one by one
    int attempt = 0, par = 0, turn = 0;
    bool keyed = false;
    int j = 1;
    while (j < npoint)
    {
        float4* const pool = pools + par * POOL_CAPACITY;
        int* const pool_place = pool_places + par * POOL_CAPACITY;
        // 1. the pool: all points whose minimum lies above `floor_bits`, at most POOL_CAPACITY
        // Every wavefront reads ROWS of its points, a row of 16 lanes each, and all 64, 16 at a time.
        constexpr int CHUNKS = TPK_WAVE / 16, PASSES = ROWS / 4;
        float4 other[CHUNKS], mine[PASSES];
        auto read_points = [&](const float4* points) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < CHUNKS; ++c)
                other[c] = points[c * 16 + lane % 16];
#pragma unroll
            for (int p = 0; p < PASSES; ++p)
                mine[p] = points[wave * ROWS + p * 4 + lane / 16];
        };
        int count = 0, floor_bits = 0;
        bool pooled = false;
        const bool paused = pause > 0 || one_by_one;
        if (paused)
            --pause;
        else
        {
            int narrow = 0, wide = 0; // gaps that gave no point, and too many
            for (int tries = 0; tries < POOL_TRIES; ++tries)
            {
                floor_bits = max(most_left - gap, 0);
                if (floor_bits >= most_left)
                    break; // nothing above zero, or more equal minima than a pool holds
                const int slot = attempt % 3;
                {
                    const int own_lane = not_hoisted(lane);
                    unsigned long long above[PPT];
                    int own = 0;
#pragma unroll
                    for (int i = 0; i < PPT; ++i)
                    {
                        above[i] = __ballot(t[i] > floor_bits);
                        own += __builtin_popcountll(above[i]);
                    }
                    if (own > 0) // (uniform over the wavefront)
                    {
                        int at = 0;
                        if (lane == 0)
                            at = atomicAdd(&pool_count[slot], own);
                        at = __builtin_amdgcn_readfirstlane(at);
                        if (at + own <= POOL_CAPACITY)
                        {
#pragma unroll
                            for (int i = 0; i < PPT; ++i)
                                if (PPT < 8 || __builtin_expect(above[i] != 0ull, 0)) // (a few of sixteen: no branch taken for the others)
                                {
                                    if (t[i] > floor_bits)
                                    {
                                        const int to = at + static_cast<int>(tpk_prefix_count(above[i]));
                                        pool[to] = make_float4(x[i], y[i], z[i], __int_as_float(t[i]));
                                        pool_place[to] = sorted_position<WAVES, GS>(i / GS, wave, i % GS, own_lane);
                                    }
                                    at += __builtin_popcountll(above[i]);
                                }
                        }
                    }
                }
                lds_barrier();
                read_points(pool);
                count = __builtin_amdgcn_readfirstlane(pool_count[slot]);
                if (tid == 0)
                    pool_count[(attempt + 2) % 3] = 0; // (the one before: everybody has read it)
                ++attempt;
                pooled = count > 0 && count <= POOL_CAPACITY;
                if (count == 0 && floor_bits == 0)
                    break; // nothing above zero
                if (pooled)
                    break;
                // the next gap: the number of points grows with the gap, and more than in proportion if it is far off
                if (count == 0)
                {
                    narrow = gap;
                    gap = wide > 0 ? narrow + (wide - narrow) / 2 : min(gap, 1 << 28) * 4;
                }
                else
                {
                    wide = gap;
                    if (count > 8 * POOL_CAPACITY)
                    {
                        // (most likely equal minima: a sample by itself tells where the largest one is)
                        gap = max(gap >> 3, 1 << 12);
                        break;
                    }
                    const float share = __builtin_amdgcn_sqrtf(static_cast<float>(POOL_TARGET) * __builtin_amdgcn_rcpf(static_cast<float>(count)));
                    const int next = __builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<float>(gap) * share));
                    gap = narrow > 0 ? max(next, narrow + (wide - narrow) / 2) : next;
                }
            }
        }
        if (pooled)
        {
            const float4* points = pool;
            const int* places = pool_place;
            const int found = count;
            if (count > TPK_WAVE) // 2. its best 64
            {
                if (wave == 0)
                {
                    // A floor that leaves at most 64, and not many fewer if that can be had: between the pool's own (more)
                    // and its largest minimum (none).
                    const int own_lane = not_hoisted(lane);
                    int v[POOL_CAPACITY / TPK_WAVE], most = INT_MIN;
                    unsigned long long kept[POOL_CAPACITY / TPK_WAVE] = {};
#pragma unroll
                    for (int u = 0; u < POOL_CAPACITY / TPK_WAVE; ++u)
                    {
                        v[u] = u * TPK_WAVE + own_lane < count ? __float_as_int(pool[u * TPK_WAVE + own_lane].w) : INT_MIN;
                        most = max(most, v[u]);
                    }
                    // (Ten halvings tell apart what lies a thousandth of the pool's range from each other.  On a lattice whose
                    // distances differ by their rounding alone they left nothing, and a sample at a time was taken instead: 4096 of
                    // 16384 points of a lattice of 100^3 3750 -> 1043 us, of 2048 points of one of 30^3 206 -> 128.)
                    int high = wave_max_to_scalar(most), low = floor_bits, share = (TPK_WAVE - 6) * 256 / count;
                    count = 0;
                    for (int tries = 0; tries < 10 || (count == 0 && high - low > 1); ++tries)
                    {
                        // (first where they would lie if they were evenly spread)
                        const int middle = high - static_cast<int>(static_cast<long long>(high - low) * share / 256);
                        share = 128;
                        unsigned long long above[POOL_CAPACITY / TPK_WAVE];
                        int have = 0;
#pragma unroll
                        for (int u = 0; u < POOL_CAPACITY / TPK_WAVE; ++u)
                        {
                            above[u] = __ballot(v[u] > middle);
                            have += __builtin_popcountll(above[u]);
                        }
                        if (have > TPK_WAVE)
                            low = middle;
                        else
                        {
                            high = middle;
                            count = have;
#pragma unroll
                            for (int u = 0; u < POOL_CAPACITY / TPK_WAVE; ++u)
                                kept[u] = above[u];
                            if (have >= TPK_WAVE - 7)
                                break;
                        }
                    }
                    int to = 0;
#pragma unroll
                    for (int u = 0; u < POOL_CAPACITY / TPK_WAVE; ++u)
                    {
                        if (v[u] > high && count > 0) // (0 left: too many are equal)
                        {
                            best[to + tpk_prefix_count(kept[u])] = pool[u * TPK_WAVE + own_lane];
                            best_place[to + tpk_prefix_count(kept[u])] = pool_place[u * TPK_WAVE + own_lane];
                        }
                        to += __builtin_popcountll(kept[u]);
                    }
                    if (lane == 0)
                        best_of = int2{count, high};
                }
                lds_barrier();
                read_points(best);
                const int2 trimmed = best_of;
                count = __builtin_amdgcn_readfirstlane(trimmed.x);
                floor_bits = __builtin_amdgcn_readfirstlane(trimmed.y);
                points = best;
                places = best_place;
            }
            if (count > 0) // (0: more equal minima at the top than a pool takes)
            {
                const unsigned long long everyone = ~0ull >> (TPK_WAVE - count);
                const int own_lane = not_hoisted(lane);
                // 3. its relation.  Point i comes before point r if it holds more (or as much, with a smaller tie key); it
                // lowers r if it is closer than what r holds, and keeps it in the pool if it is further than the floor.
                // (Bits of a ballot: four rows of 16 points.)
#pragma unroll
                for (int p = 0; p < PASSES; ++p)
                {
                    const int row = wave * ROWS + p * 4;
                    const int held = __float_as_int(mine[p].w);
                    unsigned long long before[CHUNKS], equal[CHUNKS], any_equal = 0ull;
                    const unsigned long long rows = row + 4 <= count ? ~0ull : row < count ? (1ull << (16 * (count - row))) - 1ull : 0ull;
#pragma unroll
                    for (int c = 0; c < CHUNKS; ++c)
                    {
                        const unsigned long long valid = (static_cast<unsigned long long>(static_cast<unsigned>(everyone >> (c * 16)) & 0xFFFFu) * 0x0001000100010001ull) & rows;
                        // (a point itself: bit row % 16 of its row in the chunk that holds it)
                        const unsigned long long self = row / 16 == c ? 0x0008000400020001ull << (row % 16) : 0ull;
                        const int theirs = __float_as_int(other[c].w);
                        before[c] = __ballot(theirs > held) & valid;
                        equal[c] = __ballot(theirs == held) & valid & ~self;
                        any_equal |= equal[c];
                    }
                    if (__builtin_expect(any_equal != 0, 0))
                    {
                        const unsigned key = tie_key(original_index(places[min(row + own_lane / 16, count - 1)]), log2_bs, ref_groups);
                        for (int c = 0; c < CHUNKS; ++c)
                        {
                            const unsigned theirs = tie_key(original_index(places[min(c * 16 + own_lane % 16, count - 1)]), log2_bs, ref_groups);
                            const unsigned long long first = __ballot(theirs < key);
#pragma unroll
                            for (int k = 0; k < CHUNKS; ++k)
                                before[k] |= k == c ? first & equal[k] : 0ull;
                        }
                    }
                    unsigned long long lowers[CHUNKS], stays[CHUNKS], any_stays = 0ull;
#pragma unroll
                    for (int c = 0; c < CHUNKS; ++c)
                    {
                        const int d = ordered_bits(tpk_dist2(mine[p].x, mine[p].y, mine[p].z, other[c].x, other[c].y, other[c].z));
                        TPK_WORK_ADD(row + lane / 16 < count && c * 16 + lane % 16 < count ? 1 : 0);
                        lowers[c] = __ballot(d < held) & before[c];
                        stays[c] = __ballot(d > floor_bits) & lowers[c];
                        any_stays |= stays[c];
                    }
                    // (lane r < 4 puts the 16 bits of row r of every chunk together)
                    const int shift = (own_lane % 4) * 16;
                    auto row_mask = [&](const unsigned long long (&m)[CHUNKS]) __attribute__((always_inline)) {
                        const unsigned a = static_cast<unsigned>(m[0] >> shift), b = static_cast<unsigned>(m[1] >> shift);
                        const unsigned c = static_cast<unsigned>(m[2] >> shift), d = static_cast<unsigned>(m[3] >> shift);
                        return uint2{__builtin_amdgcn_perm(b, a, 0x05040100u), __builtin_amdgcn_perm(d, c, 0x05040100u)};
                    };
                    const uint2 row_lowers = row_mask(lowers), row_before = row_mask(before);
                    if (own_lane < 4)
                    {
                        pool_blockers[row + own_lane] = row_lowers;
                        pool_before[row + own_lane] = row_before;
                    }
                    if (any_stays != 0)
                    {
                        const uint2 row_stays = row_mask(stays);
                        if (own_lane < 4 && (row_stays.x | row_stays.y) != 0)
                        {
                            pool_keepers[row + own_lane] = row_stays;
                            lds_or_u32(&keeps[par][row / 32], 1u << ((row + own_lane) % 32));
                        }
                    }
                }
                if (wave == 0 && own_lane < 2)
                    keeps[par ^ 1][own_lane] = 0; // (of the round before: everybody has read it)
                lds_barrier();
                // 4. who is taken: in the order of the pool a point is, unless one taken before it lowers it.  All points
                // whose lowering sources are decided are decided together; the first undecided one always is.
                const float4 rec = points[own_lane];
                const uint2 blockers = pool_blockers[own_lane];
                const unsigned kept_lo = keeps[par][0], kept_hi = keeps[par][1];
                unsigned long long taken = ~__ballot((blockers.x | blockers.y) != 0u) & everyone, dead = 0ull, open = everyone & ~taken;
                while (open != 0ull)
                {
                    const bool hit = ((blockers.x & static_cast<unsigned>(taken)) | (blockers.y & static_cast<unsigned>(taken >> 32))) != 0u;
                    const bool waits = ((blockers.x & static_cast<unsigned>(~dead)) | (blockers.y & static_cast<unsigned>(~dead >> 32))) != 0u;
                    const unsigned long long hits = __ballot(hit) & open, free = ~__ballot(waits) & open;
                    if ((hits | free) == 0ull)
                        break; // (cannot be: the order is strict)
                    dead |= hits;
                    taken |= free;
                    open &= ~(hits | free);
                }
                // 5. a point lowered inside the pool would be taken once the largest minimum has come down to what it holds
                // now: the round ends there
                const unsigned long long kept = static_cast<unsigned long long>(static_cast<unsigned>(__builtin_amdgcn_readfirstlane(kept_hi))) << 32 |
                                                static_cast<unsigned>(__builtin_amdgcn_readfirstlane(kept_lo));
                if (kept != 0)
                {
                    const uint2 keepers = pool_keepers[own_lane];
                    const unsigned taken_lo = static_cast<unsigned>(taken), taken_hi = static_cast<unsigned>(taken >> 32);
                    const bool lowered = ((keepers.x & taken_lo) | (keepers.y & taken_hi)) != 0u;
                    const bool out_of_it = ((blockers.x & ~keepers.x & taken_lo) | (blockers.y & ~keepers.y & taken_hi)) != 0u;
                    for (unsigned long long back = __ballot(lowered && !out_of_it) & kept; back != 0; back &= back - 1)
                    {
                        const int l = __builtin_ctzll(back);
                        const unsigned by_lo = __builtin_amdgcn_readlane(keepers.x, l), by_hi = __builtin_amdgcn_readlane(keepers.y, l);
                        const int d = ordered_bits(tpk_dist2(rec.x, rec.y, rec.z, tpk_read_lane(rec.x, l), tpk_read_lane(rec.y, l), tpk_read_lane(rec.z, l)));
                        const bool by = ((taken & (static_cast<unsigned long long>(by_hi) << 32 | by_lo)) >> lane & 1ull) != 0ull;
                        floor_bits = max(floor_bits, -wave_max_to_scalar(by ? -d : INT_MIN));
                    }
                }
                const int left = __float_as_int(rec.w);
                taken &= __ballot(left > floor_bits);
                par ^= 1;
                if (taken != 0ull) // (its first point always is)
                {
                    if (wave == 0)
                    {
                        const uint2 first = pool_before[own_lane];
                        const int number = j + __builtin_popcount(first.x & static_cast<unsigned>(taken)) + __builtin_popcount(first.y & static_cast<unsigned>(taken >> 32));
                        if (((taken >> lane) & 1ull) && number < npoint)
                            out[number] = original_index(places[lane]);
                    }
                    // the next gap: the number of points grows with the gap
                    gap = min(max(gap + (gap >> 6) * (POOL_TARGET - found), gap >> 1), 1 << 29);
                    // 6. their updates
                    j += __builtin_popcountll(taken);
                    penalty = __builtin_popcountll(taken) > 1 ? 1 : penalty;
                    most_left = floor_bits;
                    if (j < npoint)
                        update(rec.x, rec.y, rec.z, left, taken, points);
                    continue;
                }
            }
        }
        if (!paused)
        {
            pause = penalty;
            penalty = min(2 * penalty, 64);
            gap = max(gap, 1 << 12);
        }

        // One sample: every wavefront offers the best of its points (of several that hold its maximum the one with the
        // smallest tie key), and all of them find the best of those.
        int most = t[0];
#pragma unroll
        for (int i = 1; i < PPT; ++i)
            most = max(most, t[i]);
        most = wave_max_to_scalar(most);
        const int own_lane = not_hoisted(lane);
        bool several = keyed; // (where there were some there will be more)
        int held_in = 0;      // a slot that holds the maximum
        // (A wavefront whose points have all been at infinity with a sample is keyed and has nothing left: the distance there is a NaN, whose
        // bits lie below 0 and above those of -1, the minimum of points that take no part.)
        if (!keyed || most < 0)
        {
            int held = 0;
#pragma unroll
            for (int i = 0; i < PPT; ++i)
            {
                const unsigned long long holds = __ballot(t[i] == most);
                held += __builtin_popcountll(holds);
                held_in = PPT >= 8 && holds != 0ull ? i : held_in;
            }
            several = held > 1;
        }
        if (several && most >= 0)
        {
            if (!keyed)
            {
                // (from the first such round on the sort keys of this wavefront's points hold tie key and index, 14 bits each)
#pragma unroll
                for (int i = 0; i < (ORDERED ? PPT : 0); ++i)
                {
                    const int q = sorted_position<WAVES, GS>(i / GS, wave, i % GS, own_lane);
                    const int k = original_index(min(q, n - 1));
                    if (q < n)
                        sort_keys[q] = tie_key(k, log2_bs, ref_groups) << 14 | static_cast<unsigned>(k);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                keyed = true;
            }
            constexpr int BATCH = PPT < 8 ? PPT : 8;
            unsigned key = 0xFFFFFFFFu;
#pragma unroll
            for (int from = 0; from < PPT; from += BATCH)
            {
                unsigned k[BATCH];
#pragma unroll
                for (int i = 0; i < BATCH; ++i)
                {
                    const int q = min(sorted_position<WAVES, GS>((from + i) / GS, wave, (from + i) % GS, own_lane), n - 1);
                    k[i] = ORDERED ? sort_keys[q] : tie_key(q, log2_bs, ref_groups) << 14;
                }
#pragma unroll
                for (int i = 0; i < BATCH; ++i)
                    key = t[from + i] == most ? min(key, k[i] << 4 | static_cast<unsigned>(from + i)) : key;
            }
            const unsigned lowest = wave_min_u32(key);
            const int slot = static_cast<int>(lowest & 15u);
            with_slot<0, PPT>(slot, [&](auto chosen) __attribute__((always_inline)) {
                constexpr int i = chosen.value;
                if (key == lowest && t[i] == most) // (the last of 16384 points in slot 15 has the key of the lanes without one)
                {
                    offers[turn][wave] = make_float4(x[i], y[i], z[i], __int_as_float(most));
                    offer_places[turn][wave] = sorted_position<WAVES, GS>(i / GS, wave, i % GS, own_lane);
                }
            });
        }
        else
        {
            auto offer = [&](int i) __attribute__((always_inline)) {
                if (t[i] == most)
                {
                    offers[turn][wave] = make_float4(x[i], y[i], z[i], __int_as_float(most));
                    offer_places[turn][wave] = sorted_position<WAVES, GS>(i / GS, wave, i % GS, own_lane);
                }
            };
            // (sixteen tests with a branch each, of all wavefronts of a SIMD in turn, were 100 ns of such a sample's 1650: 16 x 16384 points, 4096
            // samples, even 601 -> 594 us, clusters 727 -> 724, a laser scan 868 -> 858, 4 x 16384 on a sphere 367 -> 361; where nothing is left
            // any slot that holds the maximum will do)
            if constexpr (PPT >= 8)
                with_slot<0, PPT>(held_in, [&](auto chosen) __attribute__((always_inline)) { offer(chosen.value); });
            else
            {
#pragma unroll
                for (int i = 0; i < PPT; ++i)
                    offer(i);
            }
        }
        lds_barrier();
        const float4 offer = offers[turn][lane % WAVES];
        const int place = offer_places[turn][lane % WAVES];
        turn ^= 1;
        const int gv = __builtin_amdgcn_readfirstlane(row_all_max_i32(__float_as_int(offer.w)));
        unsigned long long first = __ballot(__float_as_int(offer.w) == gv) & ((1ull << WAVES) - 1ull);
        if (gv >= 0 && (first & (first - 1)) != 0ull)
        {
            const unsigned key = (first >> lane & 1ull) != 0ull ? tie_key(original_index(place), log2_bs, ref_groups) : 0xFFFFFFFFu;
            first = __ballot(key == wave_min_u32(key)) & first;
        }
        const int w = __builtin_ctzll(first);
        float4 s = make_float4(tpk_read_lane(offer.x, w), tpk_read_lane(offer.y, w), tpk_read_lane(offer.z, w), 0.f);
        const int chosen = __builtin_amdgcn_readlane(place, w);
        if (gv < 0) // no eligible point in the whole cloud: the reference's reduction yields index 0
            s = make_float4(p0x, p0y, p0z, 0.f);
        if (tid == 0)
            out[j] = gv < 0 ? 0 : original_index(chosen);
        j += 1;
        most_left = max(gv, 0);
        update_one(s, gv < 0 ? ordered_bits(__builtin_inff()) : gv);
    }
    TPK_WORK_FLUSH
}

// Clouds that one wavefront holds, PPT points per lane: a sample at a time, 0.2 to 0.3 us each, without barriers and LDS.
// What it costs is its chain of dependent instructions.
template <int PPT>
__global__ __launch_bounds__(TPK_WAVE) void fps_wave_kernel(int n, int npoint, int log2_bs, int ref_groups,
                                                            const float* __restrict__ xyz, int32_t* __restrict__ out)
{
    xyz += static_cast<int64_t>(blockIdx.x) * n * 3;
    out += static_cast<int64_t>(blockIdx.x) * npoint;
    const int lane = threadIdx.x;
    float x[PPT], y[PPT], z[PPT];
    int t[PPT];
#pragma unroll
    for (int i = 0; i < PPT; ++i)
    {
        const int k = min(i * TPK_WAVE + lane, n - 1);
        x[i] = xyz[k * 3 + 0];
        y[i] = xyz[k * 3 + 1];
        z[i] = xyz[k * 3 + 2];
    }
#pragma unroll
    for (int i = 0; i < PPT; ++i)
        t[i] = ordered_bits(i * TPK_WAVE + lane < n && eligible(x[i], y[i], z[i]) ? 1e10f : -1.0f);
    TPK_WORK_DECL
    float sx = tpk_read_lane(x[0], 0), sy = tpk_read_lane(y[0], 0), sz = tpk_read_lane(z[0], 0);
    int mine = 0; // sample number j of the 64 not yet written, in lane j % 64
    for (int j = 1; j < npoint; ++j)
    {
        const float ux = to_vector_register(sx), uy = to_vector_register(sy), uz = to_vector_register(sz);
        int best = INT_MIN;
        TPK_WORK_ADD(PPT);
#pragma unroll
        for (int i = 0; i < PPT; ++i)
        {
            t[i] = min(t[i], ordered_bits(tpk_dist2(x[i], y[i], z[i], ux, uy, uz)));
            best = max(best, t[i]);
        }
        const int most = wave_max_to_scalar(best);
        unsigned long long holders[PPT];
        int count = 0;
#pragma unroll
        for (int i = 0; i < PPT; ++i)
        {
            holders[i] = __ballot(t[i] == most);
            count += __builtin_popcountll(holders[i]);
        }
        if (__builtin_expect(count != 1, 0))
        {
            // equal maxima: the smallest tie key
            unsigned key = 0xFFFFFFFFu;
#pragma unroll
            for (int i = 0; i < PPT; ++i)
                if (t[i] == most && i * TPK_WAVE + lane < n)
                    key = min(key, tie_key(i * TPK_WAVE + lane, log2_bs, ref_groups));
            const unsigned lowest = wave_min_u32(key);
#pragma unroll
            for (int i = 0; i < PPT; ++i)
                holders[i] = __ballot(t[i] == most && i * TPK_WAVE + lane < n && tie_key(i * TPK_WAVE + lane, log2_bs, ref_groups) == lowest);
        }
        int k = 0;
        if (most < 0)
        {
            // No eligible point in the whole cloud: the reference's reduction yields index 0.
            sx = tpk_read_lane(x[0], 0), sy = tpk_read_lane(y[0], 0), sz = tpk_read_lane(z[0], 0);
        }
        else
        {
#pragma unroll
            for (int i = 0; i < PPT; ++i)
                if (holders[i] != 0)
                {
                    const int l = __builtin_ctzll(holders[i]);
                    k = i * TPK_WAVE + l;
                    sx = tpk_read_lane(x[i], l), sy = tpk_read_lane(y[i], l), sz = tpk_read_lane(z[i], l);
                }
        }
        mine = lane == j % TPK_WAVE ? k : mine;
        if (j % TPK_WAVE == TPK_WAVE - 1)
            out[j - (TPK_WAVE - 1) + lane] = mine;
    }
    const int written = npoint / TPK_WAVE * TPK_WAVE;
    if (written + lane < npoint)
        out[written + lane] = mine;
    TPK_WORK_FLUSH
}

constexpr int FPS_CELL_WINDOW = CURVE_MAX_POINTS;            // points ordered together
constexpr int FPS_WINDOW_CELLS = FPS_CELL_WINDOW / NG_CELL;  // 256
constexpr int FPS_MAX_CELLS = 2560;                          // cells whose state fits in LDS
constexpr int FPS_CELL_POINTS = FPS_MAX_CELLS * NG_CELL;     // 163840
constexpr int FPS_LIVE_CAPACITY = (FPS_MAX_CELLS + FPS_THREADS - 1) / FPS_THREADS * TPK_WAVE; // live cells per wavefront

// Clouds too large for registers.  The cloud has been cut into windows of 16384 consecutive
// points, each ordered along the curve into 256 cells of 64 (curve_cells_kernel): records
// (x, y, z, index in the cloud) and the cells' boxes are in `sorted` / `boxes`; the running
// minima live in `temp`, in the same order (ineligible points and padding hold -1).  LDS keeps,
// for every cell, its box, its largest minimum, the tie key of the point holding it, and that
// point (x, y, z, index in the cloud).
// A minimum can only change if the new sample is closer than it, and no minimum of a cell
// exceeds the cell's largest: a cell whose box is not closer to the sample than its largest
// minimum is skipped (margin for rounding as in the register kernel), exactly.  Cell c belongs
// to wavefront c mod 16 (neighbours on the curve go to different wavefronts): the wavefront
// tests the boxes of its cells (one per lane and step), then updates the live ones - 64 points
// per cell, a few cells' loads in flight together - and renews their LDS entries.  Every wavefront then
// finds the best of its cells, and these are exchanged through LDS.
// Several samples are taken per round: the points with the largest running minima follow each other as samples
// as long as none of them changes the next one's minimum, which has to be above all that is not among them.
// Here the order is by (minimum, then the reference's tie key), which is strict - equal minima need no separate
// path - and a candidate's coordinates are at hand in LDS (the best point of its cell).  LDS also keeps every
// cell's SECOND best point's minimum and key: what a wavefront does not publish - the best points of its other
// cells, the second best of all its cells - must stay below a candidate for it to count.  A live cell is loaded
// once per round and takes the updates of all samples that reach it.
// dynamic LDS: 56 bytes per cell + FPS_LIVE_CAPACITY * 16 * 4.
constexpr int FPC_T = 16;  // samples per round at most (one wavefront decides on each)
constexpr int FPC_PUB = 2; // points a wavefront publishes per round
constexpr int FPC_CANDS = FPS_WAVES * FPC_PUB;
#ifndef FPC_CELL_BATCH_N
#define FPC_CELL_BATCH_N 4
#endif
constexpr int FPC_CELL_BATCH = FPC_CELL_BATCH_N; // live cells in flight per wavefront
static_assert(FPC_T <= FPS_WAVES && FPC_T < FPC_CANDS && FPC_PUB * FPC_CANDS <= TPK_WAVE, "one wavefront per place, one lane per pair");

// (larger minimum first, among equals the smaller tie key)
__device__ __forceinline__ bool fps_above(int v, unsigned t, int w, unsigned u)
{
    return v > w || (v == w && t < u);
}

__global__ __launch_bounds__(FPS_THREADS) void fps_cells_batched_kernel(
    int n, int npoint, int log2_bs, int groups, int cells, const float* __restrict__ xyz,
    const float4* __restrict__ sorted, const float4* __restrict__ boxes, float* __restrict__ temp,
    int32_t* __restrict__ out)
{
    extern __shared__ float4 cell_best[];                                  // [cells] x, y, z, index
    float* const box = reinterpret_cast<float*>(cell_best + cells);        // [6][cells] lo.xyz, hi.xyz
    int* const cell_max = reinterpret_cast<int*>(box + 6 * cells);         // [cells] bits of the largest minimum
    unsigned* const cell_tie = reinterpret_cast<unsigned*>(cell_max + cells); // [cells] its point's tie key
    int* const cell_max2 = reinterpret_cast<int*>(cell_tie + cells);       // [cells] the same for the second best point
    unsigned* const cell_tie2 = reinterpret_cast<unsigned*>(cell_max2 + cells);
    unsigned* const live_all = cell_tie2 + cells;                          // per wavefront: live cell | samples that reach it << 16
    __shared__ int cand_val[2][FPC_CANDS];      // published points: minimum, tie key, cell
    __shared__ unsigned cand_tie[2][FPC_CANDS];
    __shared__ int cand_cell[2][FPC_CANDS];
    __shared__ int kept_val[2][FPS_WAVES];      // per wavefront: the best of what it does not publish
    __shared__ unsigned kept_tie[2][FPS_WAVES];
    __shared__ int order[2][FPC_CANDS];         // published point of every place
    __shared__ __align__(16) float4 taken[2][FPC_T]; // x, y, z, index of the point of place k
    __shared__ int follows[2][FPC_T];           // 1: the point of place k may follow those before it
    __shared__ __align__(16) float4 lone[2][FPS_WAVES]; // rounds with one sample: every wavefront's best point

    xyz += static_cast<int64_t>(blockIdx.x) * n * 3;
    sorted += static_cast<int64_t>(blockIdx.x) * cells * NG_CELL;
    boxes += static_cast<int64_t>(blockIdx.x) * cells * NG_BOX;
    temp += static_cast<int64_t>(blockIdx.x) * cells * NG_CELL;
    out += static_cast<int64_t>(blockIdx.x) * npoint;
    const int tid = threadIdx.x;
    const int lane = tid & (TPK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / TPK_WAVE);
    unsigned* const live = live_all + wave * FPS_LIVE_CAPACITY;
    const int steps = (cells + FPS_THREADS - 1) / FPS_THREADS; // cells per lane
    const unsigned bs_mask = (1u << log2_bs) - 1u;
    auto tie_key = [&](unsigned k) __attribute__((always_inline)) {
        const unsigned rev = log2_bs ? (__brev(k & bs_mask) >> (32 - log2_bs)) : 0u;
        return rev * static_cast<unsigned>(groups) + (k >> log2_bs);
    };

    // Set-up: minima, boxes and largest minima (best points are found by the first update: it reaches every cell).
    for (int c = wave; c < cells; c += FPS_WAVES)
    {
        const float4 r = sorted[c * NG_CELL + lane];
        const bool takes_part = __float_as_int(r.w) != 0x7FFFFFFF && eligible(r.x, r.y, r.z);
        temp[c * NG_CELL + lane] = takes_part ? 1e10f : -1.0f;
        const bool any = __ballot(takes_part) != 0;
        if (lane < 6)
        {
            const float4 b = boxes[c * NG_BOX + lane / 3];
            const int a = lane % 3;
            box[lane * cells + c] = a == 0 ? b.x : a == 1 ? b.y : b.z;
        }
        if (lane == 6)
        {
            cell_max[c] = ordered_bits(any ? 1e10f : -1.0f);
            cell_tie[c] = 0xFFFFFFFFu;
            cell_max2[c] = ordered_bits(-1.0f);
            cell_tie2[c] = 0xFFFFFFFFu;
        }
    }
    const float p0x = xyz[0], p0y = xyz[1], p0z = xyz[2];
    if (tid == 0)
    {
        out[0] = 0;
        taken[0][0] = make_float4(p0x, p0y, p0z, 0.f);
    }
    __syncthreads();

    // Rounds in which only one point follows cost more this way than with one sample per round (two barriers
    // more, second bests): from the second such round in a row on, the next 1, 2, 4 .. 32 rounds take one sample
    // each, the plain way.
    int ns = 1, j = 1, pause = 0, penalty = 0;
    float4 fetched = taken[0][0]; // lane k < ns: sample k of the round before
    for (int round = 1; j < npoint; ++round)
    {
        const int par = round & 1;
        // 1. the live cells among this wavefront's, and which of the round before's samples reach each
        int count = 0;
        for (int step = 0; step < steps; ++step)
        {
            const int c = (step * TPK_WAVE + lane) * FPS_WAVES + wave;
            unsigned reach = 0;
            if (c < cells)
            {
                const float lx = box[0 * cells + c], ly = box[1 * cells + c], lz = box[2 * cells + c];
                const float hx = box[3 * cells + c], hy = box[4 * cells + c], hz = box[5 * cells + c];
                const float most = __int_as_float(cell_max[c]);
                for (int k = 0; k < ns; ++k)
                {
                    const float sx = tpk_read_lane(fetched.x, k), sy = tpk_read_lane(fetched.y, k), sz = tpk_read_lane(fetched.z, k);
                    const float dx = fmaxf(fmaxf(lx - sx, sx - hx), 0.f);
                    const float dy = fmaxf(fmaxf(ly - sy, sy - hy), 0.f);
                    const float dz = fmaxf(fmaxf(lz - sz, sz - hz), 0.f);
                    const float lb = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
                    reach |= lb * 0.999998f < most ? 1u << k : 0u;
                }
            }
            const unsigned long long mask = __ballot(reach != 0);
            if (reach != 0)
                live[count + tpk_prefix_count(mask)] = static_cast<unsigned>(c) | (reach << 16);
            count += __builtin_popcountll(mask);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();

        // 2. their points: new minima, and the cell's best and second best point
        for (int i0 = 0; i0 < count; i0 += FPC_CELL_BATCH)
        {
            unsigned entry[FPC_CELL_BATCH];
            float4 r[FPC_CELL_BATCH];
            float m[FPC_CELL_BATCH];
#pragma unroll
            for (int u = 0; u < FPC_CELL_BATCH; ++u)
            {
                entry[u] = __builtin_amdgcn_readfirstlane(live[min(i0 + u, count - 1)]);
                const int c = static_cast<int>(entry[u] & 0xFFFFu);
                r[u] = sorted[c * NG_CELL + lane];
                m[u] = temp[c * NG_CELL + lane];
            }
#pragma unroll
            for (int u = 0; u < FPC_CELL_BATCH; ++u)
            {
                if (i0 + u >= count) // wave-uniform
                    break;
                const int c = static_cast<int>(entry[u] & 0xFFFFu);
                const int old_bits = ordered_bits(m[u]);
                int new_bits = old_bits;
                for (unsigned reach = entry[u] >> 16; reach != 0; reach &= reach - 1)
                {
                    const int k = __builtin_ctz(reach);
                    const float d = tpk_dist2(r[u].x, r[u].y, r[u].z, tpk_read_lane(fetched.x, k), tpk_read_lane(fetched.y, k),
                                              tpk_read_lane(fetched.z, k));
                    new_bits = min(ordered_bits(d), new_bits); // -1 stays -1
                }
                if (new_bits != old_bits)
                    temp[c * NG_CELL + lane] = __int_as_float(new_bits);
                const unsigned k = static_cast<unsigned>(__float_as_int(r[u].w));
                const unsigned tk = tie_key(k);
                int first_val, second_val;
                const int first = winning_lane(new_bits, tk, first_val);
                const int second = winning_lane(lane == first ? INT_MIN : new_bits, tk, second_val);
                if (lane == first)
                {
                    cell_max[c] = first_val;
                    cell_tie[c] = tk;
                    cell_best[c] = make_float4(r[u].x, r[u].y, r[u].z, __int_as_float(static_cast<int>(k)));
                }
                if (lane == second)
                {
                    cell_max2[c] = second_val;
                    cell_tie2[c] = tk;
                }
            }
        }

        // 3. the two best of this wavefront's cells, and the best of what it keeps to itself: per lane the best
        // cell (b1) and the best of everything else the lane knows of (b2: its other cells' best points and all
        // its cells' second best points)
        int b1v = INT_MIN, b2v = INT_MIN, b1c = 0;
        unsigned b1t = 0xFFFFFFFFu, b2t = 0xFFFFFFFFu;
        if (pause > 0) // wave-uniform, the same in all wavefronts
        {
            for (int step = 0; step < steps; ++step)
            {
                const int c = (step * TPK_WAVE + lane) * FPS_WAVES + wave;
                if (c < cells)
                {
                    const int v = cell_max[c];
                    const unsigned t = cell_tie[c];
                    if (fps_above(v, t, b1v, b1t))
                    {
                        b1v = v;
                        b1t = t;
                        b1c = c;
                    }
                }
            }
            int v1, all_v;
            const int l1 = winning_lane(b1v, b1t, v1);
            const unsigned t1 = __builtin_amdgcn_readlane(b1t, l1);
            const float4 mine = cell_best[__builtin_amdgcn_readlane(b1c, l1)];
            if (lane == 0)
            {
                cand_val[par][wave] = v1;
                cand_tie[par][wave] = t1;
                lone[par][wave] = mine;
            }
            lds_barrier();
            const int wl = winning_lane(lane < FPS_WAVES ? cand_val[par][lane] : INT_MIN,
                                        lane < FPS_WAVES ? cand_tie[par][lane] : 0xFFFFFFFFu, all_v);
            fetched = lone[par][wl];
            if (all_v < 0) // no eligible point in the whole cloud: the reference's reduction yields index 0
                fetched = make_float4(p0x, p0y, p0z, 0.f);
            if (tid == 0)
                out[j] = __float_as_int(fetched.w);
            ns = 1;
            j += 1;
            --pause;
            continue;
        }
        for (int step = 0; step < steps; ++step)
        {
            const int c = (step * TPK_WAVE + lane) * FPS_WAVES + wave;
            if (c < cells)
            {
                const int v = cell_max[c], v2 = cell_max2[c];
                const unsigned t = cell_tie[c], t2 = cell_tie2[c];
                if (fps_above(v, t, b1v, b1t))
                {
                    b2v = b1v;
                    b2t = b1t;
                    b1v = v;
                    b1t = t;
                    b1c = c;
                }
                else if (fps_above(v, t, b2v, b2t))
                {
                    b2v = v;
                    b2t = t;
                }
                if (fps_above(v2, t2, b2v, b2t))
                {
                    b2v = v2;
                    b2t = t2;
                }
            }
        }
        {
            int v1, v2, v3 = INT_MIN;
            const int l1 = winning_lane(b1v, b1t, v1);
            const unsigned t1 = __builtin_amdgcn_readlane(b1t, l1);
            const int c1 = __builtin_amdgcn_readlane(b1c, l1);
            const int left_v = lane == l1 ? b2v : b1v;
            const unsigned left_t = lane == l1 ? b2t : b1t;
            const int l2 = winning_lane(left_v, left_t, v2);
            const unsigned t2 = __builtin_amdgcn_readlane(left_t, l2);
            const int c2 = __builtin_amdgcn_readlane(b1c, l2);
            const bool two = l2 != l1; // (else the second best is something of the first lane's: not published)
            unsigned t3 = 0xFFFFFFFFu;
            if (two)
            {
                const int rest_v = (lane == l1 || lane == l2) ? b2v : b1v;
                const unsigned rest_t = (lane == l1 || lane == l2) ? b2t : b1t;
                const int l3 = winning_lane(rest_v, rest_t, v3);
                t3 = __builtin_amdgcn_readlane(rest_t, l3);
            }
            if (lane == 0)
            {
                cand_val[par][wave * 2 + 0] = v1;
                cand_tie[par][wave * 2 + 0] = t1;
                cand_cell[par][wave * 2 + 0] = c1;
                cand_val[par][wave * 2 + 1] = two ? v2 : INT_MIN;
                cand_tie[par][wave * 2 + 1] = two ? t2 : 0xFFFFFFFFu;
                cand_cell[par][wave * 2 + 1] = two ? c2 : 0;
                kept_val[par][wave] = two ? v3 : v2;
                kept_tie[par][wave] = two ? t3 : t2;
            }
        }
        lds_barrier();

        // 4. the list is sorted out by all wavefronts together.  First every wavefront finds the places of its own
        // published points among all of them (lane (c, o): is point o above my point c?).
        {
            const int c = lane / FPC_CANDS, o = lane % FPC_CANDS;
            const int mine = wave * FPC_PUB + (c < FPC_PUB ? c : 0);
            const int mv = cand_val[par][mine], ov = cand_val[par][o];
            const unsigned mt = cand_tie[par][mine], ot = cand_tie[par][o];
            // (points that are not published are all alike: the lower number first)
            const bool higher = fps_above(ov, ot, mv, mt) || (ov == mv && ot == mt && o < mine);
            const unsigned long long above = __ballot(c < FPC_PUB && higher);
            if (o == 0 && c < FPC_PUB)
                order[par][__builtin_popcountll((above >> (c * FPC_CANDS)) & ((1ull << FPC_CANDS) - 1ull))] = mine;
        }
        lds_barrier();
        // Then wavefront k looks at the point of place k: the point of place 0 is the reference's choice; a later
        // one may follow when it is above everything unpublished and none of the points before it changes its
        // minimum (lane i: point i).
        if (wave < FPC_T)
        {
            const int at = order[par][wave], before = order[par][lane < wave ? lane : 0];
            const int val = cand_val[par][at];
            const unsigned tie = cand_tie[par][at];
            float4 rec = cell_best[cand_cell[par][at]];
            const float4 earlier = cell_best[cand_cell[par][before]];
            int kept_v;
            const int hv = lane < FPS_WAVES ? kept_val[par][lane] : INT_MIN;
            const unsigned ht = lane < FPS_WAVES ? kept_tie[par][lane] : 0xFFFFFFFFu;
            const int kl = winning_lane(hv, ht, kept_v);
            const unsigned kept_t = __builtin_amdgcn_readlane(ht, kl);
            const bool spoiled = lane < wave && ordered_bits(tpk_dist2(rec.x, rec.y, rec.z, earlier.x, earlier.y, earlier.z)) < val;
            // (its minimum must be above 0: the samples before it drop to 0 and keep their tie keys)
            const bool may = wave == 0 || (__ballot(spoiled) == 0ull && fps_above(val, tie, kept_v, kept_t) && val > 0);
            if (wave == 0 && val < 0) // no eligible point in the whole cloud: the reference's reduction yields index 0
                rec = make_float4(p0x, p0y, p0z, 0.f);
            if (lane == 0)
            {
                taken[par][wave] = rec;
                follows[par][wave] = may ? 1 : 0;
            }
        }
        lds_barrier();
        int accept = static_cast<int>(__builtin_ctzll(~__ballot(lane < FPC_T && follows[par][lane < FPC_T ? lane : 0] != 0)));
        accept = min(accept, npoint - j); // (>= 1: the point of place 0 always follows)
        if (wave == 0 && lane < accept)
            out[j + lane] = __float_as_int(taken[par][lane].w);
        fetched = taken[par][lane < accept ? lane : 0];
        ns = accept;
        j += accept;
        if (accept > 1)
            penalty = 0;
        else
        {
            pause = penalty;
            penalty = penalty ? min(2 * penalty, 32) : 1;
        }
    }
}

// Clouds too large for registers: points and running minima stream from global memory.
__global__ __launch_bounds__(FPS_THREADS) void fps_streaming_kernel(
    int n, int npoint, int log2_bs, int groups, const float* __restrict__ xyz,
    float* __restrict__ temp, int32_t* __restrict__ out)
{
    __shared__ WaveRecord records[2][FPS_WAVES];

    xyz += static_cast<int64_t>(blockIdx.x) * n * 3;
    temp += static_cast<int64_t>(blockIdx.x) * n;
    out += static_cast<int64_t>(blockIdx.x) * npoint;
    const int tid = threadIdx.x;
    const int lane = tid & (TPK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / TPK_WAVE);

    for (int k = tid; k < n; k += FPS_THREADS)
        temp[k] = 1e10f;

    const unsigned bs_mask = (1u << log2_bs) - 1u;
    const unsigned rev = log2_bs ? (__brev(tid & bs_mask) >> (32 - log2_bs)) : 0u;
    const unsigned tk_base = rev * static_cast<unsigned>(groups);

    const float p0x = xyz[0], p0y = xyz[1], p0z = xyz[2];
    float sx = p0x, sy = p0y, sz = p0z;
    if (tid == 0)
        out[0] = 0;

    for (int j = 1; j < npoint; ++j)
    {
        float best = -1.0f;
        int bk = tid < n ? tid : 0;
        for (int k = tid; k < n; k += FPS_THREADS)
        {
            const float px = xyz[k * 3 + 0], py = xyz[k * 3 + 1], pz = xyz[k * 3 + 2];
            if (!eligible(px, py, pz))
                continue;
            const float d = tpk_dist2(px, py, pz, sx, sy, sz);
            const float d2 = fminf(d, temp[k]);
            temp[k] = d2;
            bk = d2 > best ? k : bk;
            best = d2 > best ? d2 : best;
        }
        const unsigned my_tk = tk_base + (static_cast<unsigned>(bk) >> log2_bs);

        int wave_val;
        const int wl = winning_lane(ordered_bits(best), my_tk, wave_val);
        WaveRecord r;
        r.val = wave_val;
        r.tk = __builtin_amdgcn_readlane(my_tk, wl);
        r.k = __builtin_amdgcn_readlane(bk, wl);
        r.x = xyz[r.k * 3 + 0];
        r.y = xyz[r.k * 3 + 1];
        r.z = xyz[r.k * 3 + 2];
        if (lane == 0)
            records[j & 1][wave] = r;
        __syncthreads();

        int k;
        int gv_unused;
        reduce_records<FPS_WAVES>(records[j & 1], lane, p0x, p0y, p0z, k, sx, sy, sz, gv_unused);
        if (tid == 0)
            out[j] = k;
    }
}

__global__ __launch_bounds__(256) void fill_zero_i32_kernel(int32_t* p, int64_t count)
{
    int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
    for (; t < count; t += stride)
        p[t] = 0;
}

// The reference's block size for n points (cuda/include/cuda_utils.h:13-18), as a log2.
int reference_log2_block(int n)
{
    const int pow_2 = static_cast<int>(std::log(static_cast<double>(n)) / std::log(2.0));
    int v = 1 << pow_2;
    if (v > 512)
        v = 512;
    if (v < 1)
        v = 1;
    int l = 0;
    while ((1 << l) < v)
        ++l;
    return l;
}

template <int PPT, int WAVES, int GS, bool ORDERED>
int launch_pool(int b, int n, int npoint, int log2_bs, int groups, const float* xyz, int32_t* out, hipStream_t s)
{
    if (n > PPT * WAVES * TPK_WAVE || n > FPS_REGISTER_POINTS)
        return TPK_ERR_UNSUPPORTED;
    const int key_capacity = n > CURVE_BINS ? (n + 63) & ~63 : CURVE_BINS; // (the ordering borrows CURVE_BINS words)
    const size_t lds = ORDERED ? (2 * static_cast<size_t>(key_capacity) + CURVE_BINS) * sizeof(unsigned) : 0;
    auto kernel = fps_pool_kernel<PPT, WAVES, GS, ORDERED>;
    const int allowed = tpk_allow_lds(reinterpret_cast<const void*>(kernel), lds);
    if (allowed != TPK_OK)
        return allowed;
    hipLaunchKernelGGL(kernel, dim3(b), dim3(WAVES * TPK_WAVE), lds, s, n, npoint, log2_bs, groups, key_capacity,
                       xyz, out);
    return tpk_launch_status();
}

template <int PPT>
int launch_wave(int b, int n, int npoint, int log2_bs, int groups, const float* xyz, int32_t* out, hipStream_t s)
{
    if (n > PPT * TPK_WAVE)
        return TPK_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(fps_wave_kernel<PPT>, dim3(b), dim3(TPK_WAVE), 0, s, n, npoint, log2_bs, groups, xyz, out);
    return tpk_launch_status();
}

// Workspace of the cell kernel: ordered records, boxes, minima (each 256-byte aligned).
struct CellLayout
{
    int cells; // per cloud
    size_t sorted, boxes, temp, coarse, total;
};
// Clouds of more than one window are brought into a coarse order first (coarse_order.h), in batches it can index.
bool fps_coarse_first(int b, int n)
{
    return n >= CO_MIN_ROWS && static_cast<int64_t>(b) * n < (1LL << 30);
}
CellLayout cell_layout(int b, int n)
{
    auto up = [](size_t v) { return (v + 255) & ~static_cast<size_t>(255); };
    CellLayout l;
    l.cells = static_cast<int>(tpk_ceil_div(n, FPS_CELL_WINDOW)) * FPS_WINDOW_CELLS;
    const size_t all = static_cast<size_t>(b) * l.cells;
    l.sorted = 0;
    l.boxes = up(all * NG_CELL * sizeof(float4));
    l.temp = up(l.boxes + all * NG_CELL_BOXES * sizeof(float4));
    l.coarse = up(l.temp + all * NG_CELL * sizeof(float));
    l.total = fps_coarse_first(b, n) ? up(l.coarse + coarse_layout(static_cast<int64_t>(b) * n).total) : l.coarse;
    return l;
}

size_t streaming_bytes(int b, int n)
{
    return static_cast<size_t>(b) * static_cast<size_t>(n) * sizeof(float);
}

} // namespace

extern "C" size_t tpk_fps_workspace_bytes(int b, int n)
{
    if (b <= 0 || n <= FPS_REGISTER_POINTS)
        return 0;
    return n <= FPS_CELL_POINTS ? cell_layout(b, n).total : streaming_bytes(b, n);
}

extern "C" int tpk_fps_f32(int b, int n, int npoint, const float* xyz, void* workspace,
                           size_t workspace_bytes, int32_t* idx_out, void* stream)
{
    if (b < 0 || n < 0 || npoint < 0)
        return TPK_ERR_INVALID_ARG;
    if (b == 0 || npoint == 0)
        return TPK_OK;
    if (!idx_out)
        return TPK_ERR_INVALID_ARG;
    hipStream_t s = tpk_stream(stream);
    if (n == 0)
    {
        // Nothing to sample from: the reference returns its zero-initialised output.
        const int64_t count = static_cast<int64_t>(b) * npoint;
        hipLaunchKernelGGL(fill_zero_i32_kernel,
                           dim3(static_cast<unsigned>(tpk_min64(tpk_ceil_div(count, 256), 4096))),
                           dim3(256), 0, s, idx_out, count);
        return tpk_launch_status();
    }
    if (!xyz)
        return TPK_ERR_INVALID_ARG;
    if (static_cast<int64_t>(n) * 3 > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    const int log2_bs = reference_log2_block(n);
    const int groups = static_cast<int>(tpk_ceil_div(n, 1 << log2_bs));

    // Up to 256 points one wavefront (16 clouds, a quarter to half of the points sampled: 64 points 13 us, 128 17, 256 22 - 40;
    // with pools 45 - 57; eight points per lane: 512 points 118 us against 55 with pools).  Up to 1024 points pools by eight
    // wavefronts, above by sixteen (1024 points 63 / 69 us, 2048 110 / 98, 4096 187 / 159).  Up to there the cloud is taken as it comes: the
    // ordering alone is 8 us.
    if (n <= 64)
        return launch_wave<1>(b, n, npoint, log2_bs, groups, xyz, idx_out, s);
    else if (n <= 2 * 64)
        return launch_wave<2>(b, n, npoint, log2_bs, groups, xyz, idx_out, s);
    else if (n <= 4 * 64)
        return launch_wave<4>(b, n, npoint, log2_bs, groups, xyz, idx_out, s);
    else if (n <= 8 * 64)
        return launch_pool<1, 8, 1, false>(b, n, npoint, log2_bs, groups, xyz, idx_out, s);
    else if (n <= 2 * 8 * 64)
        return launch_pool<2, 8, 2, false>(b, n, npoint, log2_bs, groups, xyz, idx_out, s);
    else if (n <= 2 * 16 * 64)
        return launch_pool<2, 16, 1, true>(b, n, npoint, log2_bs, groups, xyz, idx_out, s);
    else if (n <= 4 * 16 * 64)
        return launch_pool<4, 16, 2, true>(b, n, npoint, log2_bs, groups, xyz, idx_out, s);
    else if (n <= 8 * 16 * 64)
        return launch_pool<8, 16, 2, true>(b, n, npoint, log2_bs, groups, xyz, idx_out, s);
    else if (n <= FPS_REGISTER_POINTS)
        return launch_pool<16, 16, 2, true>(b, n, npoint, log2_bs, groups, xyz, idx_out, s);
    else if (n <= FPS_CELL_POINTS && workspace && workspace_bytes >= cell_layout(b, n).total)
    {
        // Cells of 64 points in memory, their summaries in LDS.
        const CellLayout l = cell_layout(b, n);
        char* const w = static_cast<char*>(workspace);
        PointSet cloud{xyz, nullptr, static_cast<int64_t>(b) * n, n, FPS_CELL_WINDOW,
                       reinterpret_cast<float4*>(w + l.sorted), reinterpret_cast<float4*>(w + l.boxes), nullptr, nullptr};
        PointSet none{nullptr, nullptr, 0, 1, FPS_CELL_WINDOW, nullptr, nullptr, nullptr, nullptr};
        int st = TPK_OK;
        if (fps_coarse_first(b, n))
        {
            // windows that are neighbourhoods instead of samples of the whole cloud: cells half as wide
            st = launch_coarse_order(xyz, static_cast<int64_t>(b) * n, n, w + l.coarse, s);
            if (st != TPK_OK)
                return st;
            cloud.records = reinterpret_cast<const float4*>(w + l.coarse);
        }
        st = launch_curve_cells(cloud, none, nullptr, s);
        if (st != TPK_OK)
            return st;
        const size_t lds = static_cast<size_t>(l.cells) * 56 + FPS_LIVE_CAPACITY * FPS_WAVES * sizeof(unsigned);
        auto kernel = fps_cells_batched_kernel;
        st = tpk_allow_lds(reinterpret_cast<const void*>(kernel), lds);
        if (st != TPK_OK)
            return st;
        hipLaunchKernelGGL(kernel, dim3(b), dim3(FPS_THREADS), lds, s, n, npoint, log2_bs, groups, l.cells,
                           xyz, cloud.sorted, cloud.boxes, reinterpret_cast<float*>(w + l.temp), idx_out);
    }
    else
    {
        // (also serves callers that sized the workspace for the minima only)
        const size_t need = streaming_bytes(b, n);
        if (!workspace || workspace_bytes < need)
            return TPK_ERR_WORKSPACE;
        hipLaunchKernelGGL(fps_streaming_kernel, dim3(b), dim3(FPS_THREADS), 0, s, n, npoint,
                           log2_bs, groups, xyz, static_cast<float*>(workspace), idx_out);
    }
    return tpk_launch_status();
}
