// Furthest point sampling: npoint-1 dependent rounds of "update every point's distance to
// the chosen set, pick the point whose distance is largest".
//
// One workgroup (one compute unit) owns a cloud for the whole call; the rounds of a cloud
// depend on each other, so a call runs as many workgroups as there are clouds.  Three kernels
// by cloud size:
//   up to 16384 points   fps_pool_kernel: up to 18 points per lane in registers, cloud ordered along
//                        a space filling curve so that most updates can be skipped exactly; one
//                        wavefront takes dozens of samples per round from a pool (described at the kernel);
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
// Register-resident kernel with exact pruning and pools of samples, for clouds up to 16384 points.
//
// Pools.  A round takes many samples.  After its updates let the pool be all points whose running
// minimum lies above some floor; no point outside it holds more than the floor, and minima only
// fall.  So as long as the largest minimum inside the pool lies above the floor, it is the largest
// of the cloud, its point is the next sample, and only the pool's minima have to be brought up to date
// to find the one after it.  A pool of at most 64 points is a lane each of ONE wavefront, and the
// whole sequence runs in its registers: maximum over the lanes, the point's coordinates by lane
// reads, one distance per lane - a chain of 40 dependent instructions, 0.1 us, without a barrier or
// a trip to LDS.  On the clouds this was made for a pool of 44 gives about 31 samples.  (The version before
// let every wavefront offer its two best points and took those that did not change each other: 8
// samples per round, 0.37 us each; now 0.2.  Two points per lane in the pool would save two rounds of five and
// cost every step a third more.)
//
// Two kinds of wavefronts.  Wavefront 0 samples pools and holds no points.  The others hold the cloud,
// PPT points per lane; while wavefront 0 samples they bring their points up to date with the samples
// it has published so far (8 at a time, through LDS), and when it reports the end of the pool they gather
// the next one.  What share below the largest minimum makes a pool of the wanted size is carried from round
// to round; a pool that came out empty or too full is gathered again.
//
// Pruning.  A point's running minimum changes only if its distance to the new sample is smaller
// than that minimum, and no minimum exceeds the one the round's first sample held.  So a set of
// points whose bounding box is further from the sample than the square root of that value cannot
// change, and its update can be skipped without changing any result.  To make such sets exist, the
// kernel first orders the cloud along a Hilbert curve (12-bit position of its cell in a 16^3 grid,
// counting sort in LDS) and cuts the curve into cells of 64 * GS consecutive points.  A cell is GS
// registers of the 64 lanes of one wavefront; cells go round-robin to the wavefronts, so the cells around a
// sample belong to different ones.  A wavefront tests its up to 8 boxes against 8 samples at
// once, a lane per pair, and updates only what is reached (wave-uniform branches).  The fp32 box
// distance is compared with a relative margin of 2e-6, several times the rounding error of either
// side, so a skipped update is provably a no-op.
//
// Equal maxima inside a pool go by the reference's tie key.  When more points hold the same value than
// a pool takes, when nothing above zero is left, or when a coordinate is not finite (such a point never
// falls to zero), rounds take one sample by the tie key over all points holding the maximum.
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ unsigned tie_key(int k, int log2_bs, int ref_groups)
{
    const unsigned bs_mask = (1u << log2_bs) - 1u;
    const unsigned rev = log2_bs ? (__brev(static_cast<unsigned>(k) & bs_mask) >> (32 - log2_bs)) : 0u;
    return rev * static_cast<unsigned>(ref_groups) + (static_cast<unsigned>(k) >> log2_bs);
}

// The words of LDS through which the wavefronts of a workgroup agree on a round's winner.
struct RoundWords
{
    int max_val;      // atomic max of the running minima (bit patterns), starts at INT_MIN
    unsigned min_tie; // atomic min of the tie keys of the points holding max_val
};

// LDS atomics without return value, issued as written: one instruction for the active lanes
// (the compiler would otherwise wrap a same-address atomic in a loop over those lanes).
__device__ __forceinline__ unsigned lds_offset(const void* p)
{
    return static_cast<unsigned>(reinterpret_cast<unsigned long long>(
        (const __attribute__((address_space(3))) char*)p));
}
__device__ __forceinline__ void lds_atomic_max_i32(int* p, int v)
{
    asm volatile("ds_max_i32 %0, %1" ::"v"(lds_offset(p)), "v"(v) : "memory");
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

// Position on the sorted curve of member `e` of group `g` held by lane `lane` of worker `worker`.
template <int WORKERS, int GS>
__device__ __forceinline__ int sorted_position(int g, int worker, int e, int lane)
{
    return ((g * WORKERS + worker) * GS + e) * TPK_WAVE + lane;
}

constexpr int POOL_CAPACITY = 2 * TPK_WAVE; // points gathered at most; the best 64 are sampled
constexpr int POOL_TARGET = 60;
constexpr int POOL_TRIES = 8;
constexpr int POOL_BATCH = 8;   // samples published at a time: one per lane of a row of 8
constexpr int POOL_DONE = 1 << 16;

// ORDERED: the cloud is ordered along the curve and updates are pruned.  Small clouds are taken as they come: all their
// points can be brought up to date in less time than a sample takes, and the ordering alone is 8 us.
template <int PPT, int WAVES, int GS, bool ORDERED>
__global__ __launch_bounds__(WAVES* TPK_WAVE) void fps_pool_kernel(
    int n, int npoint, int log2_bs, int ref_groups, int key_capacity,
    const float* __restrict__ xyz, int32_t* __restrict__ out)
{
    constexpr int THREADS = WAVES * TPK_WAVE;
    constexpr int WORKERS = WAVES - 1;
    constexpr int NG = PPT / GS;
    static_assert(NG * GS == PPT && NG * POOL_BATCH <= TPK_WAVE, "a row of 8 lanes tests each group");
    // key_capacity keys (curve position << 20) | index in curve order, kept for the whole kernel; then, during
    // set-up, key_capacity unsorted keys and the bins of the counting sort
    extern __shared__ unsigned sort_keys[];
    unsigned* const unsorted = sort_keys + key_capacity;
    int* const bins = reinterpret_cast<int*>(unsorted + key_capacity); // CURVE_BINS words
    __shared__ int wave_totals[WAVES];
    __shared__ RoundWords words[2];
    __shared__ int cloud_box[6];      // ordered ints: min x,y,z then max x,y,z
    __shared__ __align__(16) float4 group_lo[WORKERS * NG], group_hi[WORKERS * NG]; // box of every (worker, group) cell
    __shared__ __align__(16) float4 pool[POOL_CAPACITY]; // x, y, z, sorted position of the pool's points
    __shared__ int pool_min[POOL_CAPACITY];              // their running minima
    __shared__ int pool_count[3];                   // one per attempt, in turn
    __shared__ __align__(16) float4 taken[TPK_WAVE]; // the round's samples
    // By round: how many of them stand in taken[] (POOL_DONE: there will be no more), the first one's minimum,
    // what no minimum exceeds when all their updates are made; last the exclusive or of the three.
    __shared__ __align__(16) int4 published[2];
    __shared__ int pool_best[TPK_WAVE]; // where its best 64 stand, if it holds more
    __shared__ int not_finite;

    xyz += static_cast<int64_t>(blockIdx.x) * n * 3;
    out += static_cast<int64_t>(blockIdx.x) * npoint;
    const int tid = threadIdx.x;
    const int lane = tid & (TPK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / TPK_WAVE);
    const int worker = wave - 1;
    auto original_index = [&](int position) { return ORDERED ? static_cast<int>(sort_keys[position] & 0x3FFFu) : position; };

    // ---- set-up 1 and 2: order the cloud along the curve (curve_order.h)
    if (tid < 2)
    {
        words[tid] = RoundWords{INT_MIN, 0xFFFFFFFFu};
        published[tid] = int4{0, 0, 0, 0};
    }
    if (tid < 3)
        pool_count[tid] = 0;
    if (tid == 0)
        not_finite = 0;
    if constexpr (ORDERED)
        curve_order<THREADS>(xyz, n, sort_keys, unsorted, bins, cloud_box, wave_totals);
    else
        __syncthreads();

    // ---- set-up 3: this lane's points.  The curve is cut into cells of 64 * GS consecutive
    // points; cell c belongs to worker c % WORKERS as its group c / WORKERS.  Slot i of a lane =
    // group (i / GS), member (i % GS); see sorted_position().
    float x[PPT], y[PPT], z[PPT];
    int t[PPT];
#pragma unroll
    for (int gi = 0; gi < NG; ++gi)
    {
        float lo[3] = {__builtin_inff(), __builtin_inff(), __builtin_inff()};
        float hi[3] = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
#pragma unroll
        for (int e = 0; e < GS; ++e)
        {
            const int i = gi * GS + e;
            const int q = worker >= 0 ? sorted_position<WORKERS, GS>(gi, worker, e, lane) : n;
            const int k = original_index(q < n ? q : 0);
            const float px = xyz[k * 3 + 0], py = xyz[k * 3 + 1], pz = xyz[k * 3 + 2];
            const bool ok = q < n && eligible(px, py, pz);
            if (ok && !(px - px == 0.f && py - py == 0.f && pz - pz == 0.f))
                not_finite = 1;
            x[i] = ok ? px : 0.f;
            y[i] = ok ? py : 0.f;
            z[i] = ok ? pz : 0.f;
            t[i] = ordered_bits(ok ? 1e10f : -1.0f);
            lo[0] = ok ? fminf(lo[0], px) : lo[0];
            lo[1] = ok ? fminf(lo[1], py) : lo[1];
            lo[2] = ok ? fminf(lo[2], pz) : lo[2];
            hi[0] = ok ? fmaxf(hi[0], px) : hi[0];
            hi[1] = ok ? fmaxf(hi[1], py) : hi[1];
            hi[2] = ok ? fmaxf(hi[2], pz) : hi[2];
        }
        if constexpr (!ORDERED)
            continue;
        // the cell belongs to this wavefront alone: reduce over its lanes, plain store
#pragma unroll
        for (int a = 0; a < 3; ++a)
        {
            lo[a] = ordered_int_to_float(wave_min_i32(float_to_ordered_int(lo[a])));
            hi[a] = ordered_int_to_float(wave_max_i32(float_to_ordered_int(hi[a])));
        }
        if (lane == 0 && worker >= 0)
        {
            group_lo[worker * NG + gi] = make_float4(lo[0], lo[1], lo[2], 0.f);
            group_hi[worker * NG + gi] = make_float4(hi[0], hi[1], hi[2], 0.f);
        }
    }
    __syncthreads();
    const float p0x = xyz[0], p0y = xyz[1], p0z = xyz[2];
    if (tid == 0)
    {
        out[0] = 0;
        taken[0] = make_float4(p0x, p0y, p0z, 0.f);
    }
    const bool one_by_one = __builtin_amdgcn_readfirstlane(not_finite) != 0;
    __syncthreads();
    TPK_WORK_DECL

    // The updates of samples first .. first + count - 1 (at most POOL_BATCH) of taken[]; `bound`: no running minimum
    // exceeds it.  (Bit patterns of non-negative floats throughout.)
    auto update = [&](int first, int count, int bound) __attribute__((always_inline)) {
        // row r of 8 lanes tests this wavefront's group r, its lane k against sample k
        const int k = lane % POOL_BATCH, group = lane / POOL_BATCH, cell = worker * NG + (group < NG ? group : 0);
        const float4 s = taken[first + (k < count ? k : 0)];
        if constexpr (!ORDERED)
        {
            for (int from = 0; from < count; ++from)
            {
                const float sx = to_vector_register(tpk_read_lane(s.x, from)), sy = to_vector_register(tpk_read_lane(s.y, from));
                const float sz = to_vector_register(tpk_read_lane(s.z, from));
                TPK_WORK_ADD(PPT);
#pragma unroll
                for (int i = 0; i < PPT; ++i)
                    t[i] = min(t[i], ordered_bits(tpk_dist2(x[i], y[i], z[i], sx, sy, sz)));
            }
            return;
        }
        const float4 lo = group_lo[cell], hi = group_hi[cell];
        const float dx = fmaxf(fmaxf(lo.x - s.x, s.x - hi.x), 0.f);
        const float dy = fmaxf(fmaxf(lo.y - s.y, s.y - hi.y), 0.f);
        const float dz = fmaxf(fmaxf(lo.z - s.z, s.z - hi.z), 0.f);
        const float lb = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz)) * 0.999998f;
        // an empty box gives lb = +inf (never live); NaN compares false -> live
        const unsigned long long live = __ballot(k < count && group < NG && !(lb >= __int_as_float(bound)));
#pragma unroll
        for (int gi = 0; gi < NG; ++gi)
            for (unsigned reach = static_cast<unsigned>(live >> (gi * POOL_BATCH)) & 0xFFu; reach != 0; reach &= reach - 1)
            {
                const int from = __builtin_ctz(reach); // (lanes 0 .. 7 hold samples 0 .. 7)
                const float sx = to_vector_register(tpk_read_lane(s.x, from)), sy = to_vector_register(tpk_read_lane(s.y, from));
                const float sz = to_vector_register(tpk_read_lane(s.z, from));
                TPK_WORK_ADD(GS);
#pragma unroll
                for (int e = 0; e < GS; ++e)
                {
                    const int i = gi * GS + e;
                    t[i] = min(t[i], ordered_bits(tpk_dist2(x[i], y[i], z[i], sx, sy, sz)));
                }
            }
    };
    if (worker >= 0)
        update(0, 1, ordered_bits(__builtin_inff()));

    int most_left = 0;       // no running minimum exceeds this
    float gap = 0.1f;        // the pool takes what lies within this share below it
    int pause = 1, penalty = 1; // rounds to take one by one; the first finds the largest minimum
    int which = 0, attempt = 0, round = 0;
    int j = 1;
    while (j < npoint)
    {
        // 1. the pool: all points whose minimum lies above `floor_bits`, at most 64
        int count = 0, floor_bits = 0;
        bool pooled = false;
        const bool paused = pause > 0 || one_by_one;
        if (paused)
            --pause;
        else
            for (int tries = 0; tries < POOL_TRIES && !pooled; ++tries)
            {
                floor_bits = ordered_bits(fmaxf(__int_as_float(most_left) * (1.0f - gap), 0.f));
                if (floor_bits >= most_left)
                    break; // nothing above zero, or more equal minima than a pool holds
                const int slot = attempt % 3;
                if (worker >= 0)
                {
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
                                if (above[i] != 0)
                                {
                                    if (t[i] > floor_bits)
                                    {
                                        const int to = at + static_cast<int>(tpk_prefix_count(above[i]));
                                        pool[to] = make_float4(x[i], y[i], z[i], __int_as_float(sorted_position<WORKERS, GS>(i / GS, worker, i % GS, lane)));
                                        pool_min[to] = t[i];
                                    }
                                    at += __builtin_popcountll(above[i]);
                                }
                        }
                    }
                }
                lds_barrier();
                count = __builtin_amdgcn_readfirstlane(pool_count[slot]);
                if (tid == 0)
                    pool_count[(attempt + 2) % 3] = 0; // (the one before: everybody has read it)
                ++attempt;
                pooled = count > 0 && count <= POOL_CAPACITY;
                if (count == 0 && floor_bits == 0)
                    break; // nothing above zero
                const float wanted = count == 0 ? 2.0f : static_cast<float>(POOL_TARGET) / static_cast<float>(count);
                gap *= pooled ? fminf(fmaxf(wanted, 0.5f), 2.0f) : fmaxf(wanted, 0.02f);
            }
        if (pooled)
        {
            const int par = round & 1;
            int taken_now = 0; // (none: more than 64 hold the largest minimum)
            ++round;
            if (wave == 0)
            {
                // 2a. the samples, one after the other (what a step costs is its instructions, a chain of dependent
                // ones; the others' work goes into its gaps).  A point taken falls to zero, so a step takes a new one.
                __builtin_amdgcn_s_setprio(3);
                int at = lane < count ? lane : 0, left = lane < count ? pool_min[lane] : INT_MIN;
                int number = -1; // this lane's point was the number-th to be taken
                if (count > TPK_WAVE)
                {
                    // a floor that leaves at most 64, and not many fewer if that can be had: between the pool's own (more)
                    // and its largest minimum (none), first where they would lie if they were evenly spread
                    const int second = lane + TPK_WAVE < count ? pool_min[lane + TPK_WAVE] : INT_MIN;
                    int high = wave_max_to_scalar(max(left, second)), low = floor_bits;
                    unsigned long long first_ones = 0ull, second_ones = 0ull;
                    int share = (TPK_WAVE - 4) * 256 / count;
                    for (int tries = 0; tries < 6; ++tries)
                    {
                        const int middle = high - static_cast<int>(static_cast<long long>(high - low) * share / 256);
                        const unsigned long long f = __ballot(left > middle), g = __ballot(second > middle);
                        const int have = __builtin_popcountll(f) + __builtin_popcountll(g);
                        if (have > TPK_WAVE)
                            low = middle;
                        else
                        {
                            high = middle;
                            first_ones = f;
                            second_ones = g;
                            if (have >= TPK_WAVE - 12)
                                break;
                        }
                        share = 128;
                    }
                    floor_bits = high;
                    count = __builtin_popcountll(first_ones) + __builtin_popcountll(second_ones); // 0: too many are equal
                    if (left > floor_bits && count > 0)
                        pool_best[tpk_prefix_count(first_ones)] = lane;
                    if (second > floor_bits && count > 0)
                        pool_best[__builtin_popcountll(first_ones) + tpk_prefix_count(second_ones)] = lane + TPK_WAVE;
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    at = lane < count ? pool_best[lane] : 0;
                    left = lane < count ? pool_min[at] : INT_MIN;
                }
                const float4 rec = pool[at];
                int most = wave_max_to_scalar(left), now = 0;
                const int top = most;
                if (lane == 0)
                    published[par ^ 1] = int4{0, 0, 0, 0}; // (the round before: everybody has left it)
                auto publish = [&](int from, int flags) __attribute__((always_inline)) {
                    if (number >= from)
                        taken[number] = rec;
                    // (a wavefront's LDS accesses are executed in order: nothing to wait for)
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    if (lane == 0)
                        published[par] = int4{now | flags, top, floor_bits, (now | flags) ^ top ^ floor_bits};
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                };
                while (true)
                {
                    const int from = now;
#pragma unroll
                    for (int u = 0; u < POOL_BATCH; ++u)
                        if (__builtin_expect(most > floor_bits, 1))
                        {
                            unsigned long long holders = __ballot(left == most);
                            if (__builtin_expect(__builtin_popcountll(holders) != 1, 0))
                            {
                                const unsigned key = left == most ? tie_key(original_index(__float_as_int(rec.w)), log2_bs, ref_groups) : 0xFFFFFFFFu;
                                holders = __ballot(key == wave_min_u32(key));
                            }
                            const int l = __builtin_ctzll(holders);
                            const float d = tpk_dist2(rec.x, rec.y, rec.z, tpk_read_lane(rec.x, l), tpk_read_lane(rec.y, l), tpk_read_lane(rec.z, l));
                            number = lane == l ? now : number;
                            left = min(left, ordered_bits(d));
                            ++now;
                            most = wave_max_to_scalar(left);
                        }
                    if (most <= floor_bits)
                    {
                        publish(from, POOL_DONE);
                        break;
                    }
                    publish(from, 0);
                }
                __builtin_amdgcn_s_setprio(0);
                if (number >= 0 && j + number < npoint)
                    out[j + number] = original_index(__float_as_int(rec.w));
                taken_now = now;
            }
            else
            {
                // 2b. meanwhile the updates of the samples published so far
                const volatile int4* const word = &published[par];
                int seen = 0;
                while (true)
                {
                    const int state = __builtin_amdgcn_readfirstlane(word->x), top = __builtin_amdgcn_readfirstlane(word->y);
                    const int floor_now = __builtin_amdgcn_readfirstlane(word->z);
                    if ((state ^ top ^ floor_now) != __builtin_amdgcn_readfirstlane(word->w))
                        continue; // (read while it was being written)
                    floor_bits = floor_now;
                    const int ready = state & (POOL_DONE - 1);
                    if (seen < ready)
                    {
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                        for (; seen < ready; seen = min(seen + POOL_BATCH, ready))
                            update(seen, min(POOL_BATCH, ready - seen), top);
                    }
                    else if ((state & POOL_DONE) == 0)
                        __builtin_amdgcn_s_sleep(1);
                    if (state & POOL_DONE)
                        break;
                }
                taken_now = seen;
            }
            if (taken_now > 0)
            {
                j += taken_now;
                penalty = taken_now > 1 ? 1 : penalty;
                most_left = floor_bits;
                continue;
            }
        }
        if (!paused)
        {
            pause = penalty;
            penalty = min(2 * penalty, 32);
            gap = 0.02f;
        }

        // More equal minima at the top than a pool holds, or nothing above zero: one sample by the reference's tie key
        // over all points that hold the maximum (the key comes from the original index kept in the sort keys).
        if (tid == 0)
            words[which ^ 1] = RoundWords{INT_MIN, 0xFFFFFFFFu}; // (for the next time)
        if (worker >= 0)
        {
            int best = t[0];
#pragma unroll
            for (int i = 1; i < PPT; ++i)
                best = max(best, t[i]);
            const int row_best = row_all_max_i32(best);
            if ((lane & 15) == 0)
                lds_atomic_max_i32(&words[which].max_val, row_best);
        }
        lds_barrier();
        const int gv = __builtin_amdgcn_readfirstlane(words[which].max_val);
        if (gv < 0)
        {
            // No eligible point in the whole cloud: the reference's reduction yields index 0.
            if (tid == 0)
            {
                taken[0] = make_float4(p0x, p0y, p0z, 0.f);
                out[j] = 0;
            }
        }
        else
        {
            unsigned my_tk = 0xFFFFFFFFu;
            int my_q = 0;
            if (worker >= 0)
            {
#pragma unroll
                for (int i = 0; i < PPT; ++i)
                {
                    const int q = sorted_position<WORKERS, GS>(i / GS, worker, i % GS, lane);
                    if (t[i] == gv && q < n)
                    {
                        const unsigned tk = tie_key(original_index(q), log2_bs, ref_groups);
                        if (tk < my_tk)
                        {
                            my_tk = tk;
                            my_q = q;
                        }
                    }
                }
                if (my_tk != 0xFFFFFFFFu)
                    atomicMin(&words[which].min_tie, my_tk);
            }
            lds_barrier();
            if (worker >= 0 && my_tk == words[which].min_tie) // tie keys are distinct: exactly one lane
            {
                const int k = original_index(my_q);
                taken[0] = make_float4(xyz[k * 3 + 0], xyz[k * 3 + 1], xyz[k * 3 + 2], __int_as_float(my_q));
                out[j] = k;
            }
        }
        lds_barrier();
        which ^= 1;
        j += 1;
        most_left = max(gv, 0);
        if (worker >= 0)
            update(0, 1, gv < 0 ? ordered_bits(__builtin_inff()) : gv);
        lds_barrier(); // (taken[] may be written again)
    }
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
    if (n > PPT * (WAVES - 1) * TPK_WAVE || n > FPS_REGISTER_POINTS)
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
    l.temp = up(l.boxes + all * NG_BOX * sizeof(float4));
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

    // Up to 16384 points: registers of the workers of a workgroup, with one wavefront more that samples.  Sixteen
    // wavefronts throughout (eight with twice the points each: 4 - 20 us more), cells of 64 to 192 points.  Measured with a
    // quarter of the points sampled (16 clouds; the version before): 400 points 45 us (68), 1024 82 (114), 2048 134 (204),
    // 4096 234 (359), 8192 430 (768), 16384 843 (1293).
    if (n <= 15 * 64)
        return launch_pool<1, 16, 1, false>(b, n, npoint, log2_bs, groups, xyz, idx_out, s);
    else if (n <= 2 * 15 * 64)
        return launch_pool<2, 16, 2, true>(b, n, npoint, log2_bs, groups, xyz, idx_out, s);
    else if (n <= 4 * 15 * 64)
        return launch_pool<4, 16, 2, true>(b, n, npoint, log2_bs, groups, xyz, idx_out, s);
    else if (n <= 6 * 15 * 64)
        return launch_pool<6, 16, 3, true>(b, n, npoint, log2_bs, groups, xyz, idx_out, s);
    else if (n <= 12 * 15 * 64)
        return launch_pool<12, 16, 3, true>(b, n, npoint, log2_bs, groups, xyz, idx_out, s);
    else if (n <= FPS_REGISTER_POINTS)
        return launch_pool<18, 16, 3, true>(b, n, npoint, log2_bs, groups, xyz, idx_out, s);
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
