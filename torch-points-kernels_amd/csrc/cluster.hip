// Clusters grown over a neighbour matrix: the device side of grow_proximity / region_grow
// (reference: torch_points_kernels/cluster.py:9-45, where the matrix is copied to the host and a
// numba routine walks it).
//
// The reference takes the points in index order; an unseen point i starts a cluster that
// receives every unseen point reachable from i along rows of the matrix (a row lists the
// neighbours of its point and ends at the first -1).  Rows cut at nsample entries make the
// relation one-directional, so these are not connected components.  What decides the cluster of
// a point v is the smallest index among the points that reach v (v included): that point is
// reached by no smaller one, so it is unseen at its turn and starts a cluster, and every other
// point that reaches v comes later.  The labels are therefore the fixed point of
//     label[v] = min(v, label[u] for every row u that lists v),
// which is found here in two steps.  Points that list each other (all of them, where no row was
// cut) are first merged into groups by union-find: they reach and are reached by the same points.
// Then repeated sweeps hand labels from group to group with atomicMin, shortened by following
// the label of a label (valid because reaching is transitive).  Without the merging a label
// would cross a cluster one row per sweep.  Clusters are numbered by their first point, as in
// the reference, and those below min_cluster_size are dropped.
//
// Members inside a cluster, two orders:
//   TPK_MEMBERS_AS_REFERENCE  the order in which the reference's stack walk appends them.  The walk
//       of a cluster never leaves it (anything a member reaches outside was seen by an earlier
//       cluster), so the clusters are walked independently, one wavefront each; inside a cluster
//       the walk is the reference's, serial, one expanded point per step.
//   TPK_MEMBERS_BY_INDEX      ascending index: a stable radix sort (rocPRIM) of the point numbers by
//       cluster number.  Everything is data-parallel.
//
// The entry point blocks the host: the number of sweeps and the sizes of the outputs depend on
// the data.
//
// The reference's member order has a second path, tpk_grow_components / tpk_grow_rows, for callers
// with host threads at hand (the Python layer's): a stack walk is a chain of dependent steps, 0.8 us
// each on the device (row load, compare-and-swap, stack load: three trips to the L2) and 10-20 ns on
// a host core whose cache holds the cluster's rows.  The device cuts the problem into pieces that no
// entry crosses and lays each out as one compact block, the host walks the blocks side by side.
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "cloud_ids.h"
#include "grow_table.h"
#include "tpk_device.h"

namespace
{

constexpr int CL_THREADS = 256;
constexpr int CL_ROW_LANES = 16; // lanes that share one row of the matrix in a sweep
constexpr int CL_SWEEPS = 8;     // sweeps enqueued between two looks at the `changed` flags
constexpr int CL_FOLLOW = 16;    // labels followed per point and sweep
constexpr int64_t CL_MAX_POINTS = (int64_t)1 << 30;

using u64 = unsigned long long;

__global__ void __launch_bounds__(CL_THREADS)
    cluster_init_kernel(int n, int words, int* parent, int* label, int* size, int* handed, unsigned* mutual, int* changed)
{
    const int v = blockIdx.x * CL_THREADS + threadIdx.x;
    if (v < n)
    {
        parent[v] = v;
        label[v] = v;
        size[v] = 0;
        handed[v] = n; // nothing handed over yet
        for (int w = 0; w < words; ++w)
            mutual[(int64_t)v * words + w] = 0;
    }
    if (v < CL_SWEEPS)
        changed[v] = 0;
}

__global__ void __launch_bounds__(CL_THREADS) cluster_clear_kernel(int* changed)
{
    if (threadIdx.x < CL_SWEEPS)
        changed[threadIdx.x] = 0;
}

// The part of a row that counts: lanes of a group of CL_ROW_LANES hold consecutive entries (-1
// beyond the row's width); returns how many of them come before the row's end and whether the
// row ends in this chunk.
__device__ __forceinline__ int entries_before_end(int64_t nei, int shift, bool* row_ends)
{
    const unsigned ends = (unsigned)(__ballot(nei == -1) >> shift) & 0xffffu;
    *row_ends = ends != 0;
    return ends ? __builtin_ctz(ends) : CL_ROW_LANES;
}

// Bit j of a point's mask: entry j of its row is a point whose own row lists this point back.
// The smallest such point below u becomes u's first parent (a plain store: only u's lanes
// write parent[u] in this kernel), which leaves far fewer trees for the merge sweeps to hang.
__global__ void __launch_bounds__(CL_THREADS)
    cluster_mutual_kernel(int n, int nsample, int words, const int64_t* __restrict__ neighbours, unsigned* mutual,
                          int* parent)
{
    const int64_t t = (int64_t)blockIdx.x * CL_THREADS + threadIdx.x;
    const int64_t point = t / CL_ROW_LANES;
    const int g = (int)(t % CL_ROW_LANES);
    if (point >= n)
        return; // the whole group of lanes leaves together
    const int u = (int)point;
    const int shift = (int)(tpk_lane_id() & (TPK_WAVE - CL_ROW_LANES)); // first lane of this row's group
    int lowest = u;
    for (int first = 0; first < nsample; first += CL_ROW_LANES)
    {
        const int j = first + g;
        const int64_t nei = j < nsample ? neighbours[(int64_t)u * nsample + j] : -1;
        bool row_ends;
        const int valid = entries_before_end(nei, shift, &row_ends);
        bool back = false;
        if (g < valid && nei >= 0 && nei < n && nei != u)
        {
            const int64_t* other = neighbours + nei * nsample;
            for (int i = 0; i < nsample; ++i)
            {
                const int64_t e = other[i];
                if (e == -1)
                    break;
                if (e == u)
                {
                    back = true;
                    break;
                }
            }
        }
        const unsigned bits = (unsigned)(__ballot(back) >> shift) & 0xffffu;
        if (g == 0 && bits)
            atomicOr(&mutual[(int64_t)u * words + (first >> 5)], bits << (first & 31));
        if (back && (int)nei < lowest)
            lowest = (int)nei;
        if (row_ends)
            break;
    }
    // minimum over the group's lanes (the lanes of a group are together again here)
    for (int step = 1; step < CL_ROW_LANES; step <<= 1)
        lowest = min(lowest, __shfl_xor(lowest, step, CL_ROW_LANES));
    if (g == 0 && lowest < u)
        parent[u] = lowest;
}

__device__ __forceinline__ int find_root(const int* parent, int v)
{
    for (int up = parent[v]; up < v; up = parent[v])
        v = up;
    return v;
}

// Points that list each other reach the same points and are reached by the same points, so they
// can be merged outright: union-find over the mutual entries (the tree of the larger root is hung
// under the smaller root), repeated until no tree is hung any more.  Each mutual pair is handled
// from its smaller point.
__global__ void __launch_bounds__(CL_THREADS)
    cluster_merge_kernel(int n, int nsample, int words, const int64_t* __restrict__ neighbours,
                         const unsigned* __restrict__ mutual, int* parent, int* changed, int sweep)
{
    if (sweep > 0 && changed[sweep - 1] == 0)
        return;
    const int64_t t = (int64_t)blockIdx.x * CL_THREADS + threadIdx.x;
    const int64_t point = t / CL_ROW_LANES;
    const int g = (int)(t % CL_ROW_LANES);
    if (point >= n)
        return;
    const int u = (int)point;
    const int mine = find_root(parent, u);
    bool hung = false;
    for (int j = g; j < nsample; j += CL_ROW_LANES)
    {
        if (((mutual[(int64_t)u * words + (j >> 5)] >> (j & 31)) & 1u) == 0)
            continue;
        const int nei = (int)neighbours[(int64_t)u * nsample + j];
        if (nei < u)
            continue;
        const int theirs = find_root(parent, nei);
        if (theirs != mine)
        {
            // Many entries join the same two trees; only while the higher root still is a root
            // is it worth an atomic on that one address.  Otherwise another entry has hung it
            // meanwhile and this pair is looked at again in the next sweep.
            const int low = min(mine, theirs), high = max(mine, theirs);
            if (__hip_atomic_load(&parent[high], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == high)
                hung |= atomicMin(&parent[high], low) > low;
            else
                hung = true;
        }
    }
    if (g == 0 && mine < parent[u])
        atomicMin(&parent[u], mine);
    if (hung)
        changed[sweep] = 1;
}

// Shortens the trees before a merge sweep: every point moves its parent a few steps up (only
// the point's own thread writes its entry in this kernel).
__global__ void __launch_bounds__(CL_THREADS) cluster_jump_kernel(int n, int* parent, const int* changed, int sweep)
{
    if (sweep > 0 && changed[sweep - 1] == 0)
        return;
    const int v = blockIdx.x * CL_THREADS + threadIdx.x;
    if (v >= n)
        return;
    const int first = parent[v];
    int p = first;
    for (int step = 0; step < CL_FOLLOW; ++step)
    {
        const int up = parent[p];
        if (up >= p)
            break;
        p = up;
    }
    if (p < first)
        parent[v] = p;
}

// parent[v] becomes the smallest point of v's merged group.
__global__ void __launch_bounds__(CL_THREADS) cluster_flatten_kernel(int n, int* parent)
{
    const int v = blockIdx.x * CL_THREADS + threadIdx.x;
    if (v < n)
    {
        const int root = find_root(parent, v);
        if (root < parent[v])
            atomicMin(&parent[v], root);
    }
}

// One sweep over all entries.  Labels live at the first point of every merged group (`group`):
// label[group[v]] is a point that reaches v.  Every point hands the smallest label it can find by
// following its own (label of the group of the label ...) to the groups of the points its row
// lists - unless that is what it handed over last time (`handed`): labels only fall, so those
// groups still hold it or less.  Sweep `sweep` of a batch does nothing when the one before
// changed nothing, so a batch can be enqueued without looking at the flags in between.
__global__ void __launch_bounds__(CL_THREADS)
    cluster_sweep_kernel(int n, int nsample, const int64_t* __restrict__ neighbours, const int* __restrict__ group,
                         int* label, int* handed, int* changed, int sweep)
{
    if (sweep > 0 && changed[sweep - 1] == 0)
        return;
    const int64_t t = (int64_t)blockIdx.x * CL_THREADS + threadIdx.x;
    const int64_t point = t / CL_ROW_LANES;
    const int g = (int)(t % CL_ROW_LANES);
    if (point >= n)
        return; // the whole group of lanes leaves together
    const int u = (int)point;
    const int shift = (int)(tpk_lane_id() & (TPK_WAVE - CL_ROW_LANES)); // first lane of this row's group
    const int home = group[u];
    const int mine = label[home];
    const int before = handed[u];
    // A few steps upstream: any point found this way reaches u, and storing it makes the next
    // sweep's steps that much longer, so chains shorten geometrically.
    int root = mine;
    for (int step = 0; step < CL_FOLLOW; ++step)
    {
        const int up = label[group[root]];
        if (up >= root)
            break;
        root = up;
    }
    if (root == before)
        return;
    bool lowered = false;
    if (g == 0)
    {
        handed[u] = root;
        if (root < mine)
            lowered = atomicMin(&label[home], root) > root;
    }
    for (int first = 0; first < nsample; first += CL_ROW_LANES)
    {
        const int j = first + g;
        const int64_t nei = j < nsample ? neighbours[(int64_t)u * nsample + j] : -1;
        bool row_ends;
        const int valid = entries_before_end(nei, shift, &row_ends);
        if (g < valid && nei >= 0 && nei < n)
        {
            const int there = group[nei];
            if (there != home && label[there] > root)
                lowered |= atomicMin(&label[there], root) > root;
        }
        if (row_ends)
            break;
    }
    if (lowered)
        changed[sweep] = 1;
}

// Every point takes the label of its group.  Labels of other points than the first of a group
// are read by nobody, so this can be done in place.
__global__ void __launch_bounds__(CL_THREADS) cluster_spread_kernel(int n, const int* __restrict__ group, int* label)
{
    const int v = blockIdx.x * CL_THREADS + threadIdx.x;
    if (v < n && group[v] != v)
        label[v] = label[group[v]];
}

// Members per cluster, counted at the cluster's first point.  Lanes with the same label add once.
__global__ void __launch_bounds__(CL_THREADS) cluster_count_kernel(int n, const int* __restrict__ label, int* size)
{
    const int v = blockIdx.x * CL_THREADS + threadIdx.x;
    const int l = v < n ? label[v] : -1;
    u64 left = __ballot(l >= 0);
    while (left)
    {
        const int leader = __builtin_ctzll(left);
        const int which = __builtin_amdgcn_readlane(l, leader);
        const u64 same = __ballot(l == which);
        if ((int)tpk_lane_id() == leader)
            atomicAdd(&size[which], __builtin_popcountll(same));
        left &= ~same;
    }
}

// Scan input: for the first point of a kept cluster (1 << 32 | members), else 0; one more zero
// at the end so that the exclusive scan also gives the totals.
__global__ void __launch_bounds__(CL_THREADS)
    cluster_kept_kernel(int n, int min_size, const int* __restrict__ label, const int* __restrict__ size, u64* packed)
{
    const int v = blockIdx.x * CL_THREADS + threadIdx.x;
    if (v > n)
        return;
    u64 p = 0;
    if (v < n && label[v] == v && size[v] >= min_size)
        p = ((u64)1 << 32) | (unsigned)size[v];
    packed[v] = p;
}

// From the scan: number and first output position of every kept cluster.
__global__ void __launch_bounds__(CL_THREADS)
    cluster_describe_kernel(int n, const u64* __restrict__ packed, const u64* __restrict__ scanned, int* number,
                            int* seeds, int64_t* starts)
{
    const int v = blockIdx.x * CL_THREADS + threadIdx.x;
    if (v > n)
        return;
    const u64 s = scanned[v];
    const int c = (int)(s >> 32);
    const int64_t at = (int64_t)(s & 0xffffffffu);
    if (v == n)
    {
        starts[c] = at; // totals: one past the last cluster
        return;
    }
    if (packed[v] != 0)
    {
        number[v] = c;
        seeds[c] = v;
        starts[c] = at;
    }
    else
        number[v] = -1;
}

// ---- a stable sort by small keys -----------------------------------------------------------------
// Clusters, pieces and labels are few, and what has to be sorted is point numbers that stand in order: one
// counting pass over `bins` keys does it - a histogram per block of 2048 points, a prefix sum over
// (key, block), a placement that keeps the order.  3 launches, 26 us for 300000 points and 150 keys, where the
// merge sort rocPRIM picks at this size takes 20 launches and 105 us; it stays for more keys than the
// tables are made for.
constexpr int CS_WAVES = 4;
constexpr int CS_STEPS = 8;
constexpr int CS_BLOCK = CS_WAVES * CS_STEPS * TPK_WAVE;
constexpr int CS_BINS = 1024;
constexpr int CS_SCAN_THREADS = 1024;
constexpr int CS_SCAN_ROWS = 32;        // entries of a thread of the prefix sum at a time
constexpr int64_t CS_TABLE = 1 << 18; // (key, block) pairs the one workgroup of the prefix sum goes through

// The number of the point's cluster, `clusters` for points of dropped clusters.
struct ClusterKeys
{
    int clusters;
    const int* label;
    const int* number;
    __device__ __forceinline__ unsigned operator()(int v) const
    {
        const int c = number[label[v]];
        return c < 0 ? (unsigned)clusters : (unsigned)c;
    }
};

template <typename Keys>
__global__ void __launch_bounds__(CS_WAVES * TPK_WAVE) counting_histogram_kernel(int n, int bins, Keys key_of, unsigned* keys, unsigned* table)
{
    __shared__ unsigned count[CS_BINS];
    for (int k = threadIdx.x; k < bins; k += CS_WAVES * TPK_WAVE)
        count[k] = 0;
    __syncthreads();
    const int begin = blockIdx.x * CS_BLOCK;
    for (int i = begin + threadIdx.x; i < n && i < begin + CS_BLOCK; i += CS_WAVES * TPK_WAVE)
    {
        const unsigned k = key_of(i);
        keys[i] = k;
        atomicAdd(&count[k], 1u);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < bins; k += CS_WAVES * TPK_WAVE)
        table[(int64_t)k * gridDim.x + blockIdx.x] = count[k];
}

// Exclusive prefix sum of the table in place, one workgroup: a wavefront takes CS_SCAN_ROWS rows of 64 consecutive entries of a
// tile, all requested before the first is used and summed row by row.  (Bound by latency and by the lines a load touches: 16600
// entries, a run of consecutive ones per thread, one after the other, 13 to 18 us; by rows 5.2.)
__global__ void __launch_bounds__(CS_SCAN_THREADS) counting_scan_kernel(int entries, unsigned* table)
{
    __shared__ int waves[CS_SCAN_THREADS / TPK_WAVE];
    const int wave = threadIdx.x / TPK_WAVE, lane = threadIdx.x % TPK_WAVE;
    int carry = 0;
    for (int tile = 0; tile < entries; tile += CS_SCAN_THREADS * CS_SCAN_ROWS)
    {
        const int begin = tile + wave * TPK_WAVE * CS_SCAN_ROWS + lane;
        int v[CS_SCAN_ROWS];
        int sum = 0; // of the rows so far
        if (begin - lane < entries) // (wave-uniform)
        {
#pragma unroll
            for (int i = 0; i < CS_SCAN_ROWS; ++i)
                v[i] = begin + i * TPK_WAVE < entries ? (int)table[begin + i * TPK_WAVE] : 0;
#pragma unroll
            for (int i = 0; i < CS_SCAN_ROWS; ++i)
            {
                const int before = wave_exclusive_sum(v[i]);
                const int row = __builtin_amdgcn_readlane(before + v[i], TPK_WAVE - 1);
                v[i] = sum + before;
                sum += row;
            }
        }
        __syncthreads(); // (the tile before has been read)
        if (lane == 0)
            waves[wave] = sum;
        __syncthreads();
        int before = carry;
        for (int w = 0; w < CS_SCAN_THREADS / TPK_WAVE; ++w)
        {
            before += w < wave ? waves[w] : 0;
            carry += waves[w];
        }
#pragma unroll
        for (int i = 0; i < CS_SCAN_ROWS; ++i)
            if (begin + i * TPK_WAVE < entries)
                table[begin + i * TPK_WAVE] = (unsigned)(before + v[i]);
    }
}

__global__ void __launch_bounds__(CS_WAVES * TPK_WAVE)
    counting_place_kernel(int n, int bins, int bits, const unsigned* __restrict__ keys, const unsigned* __restrict__ table,
                          unsigned* __restrict__ keys_out, unsigned* __restrict__ values_out)
{
    __shared__ unsigned next[CS_WAVES][CS_BINS];
    const int wave = threadIdx.x / TPK_WAVE, lane = threadIdx.x % TPK_WAVE;
    for (int k = threadIdx.x; k < CS_WAVES * CS_BINS; k += CS_WAVES * TPK_WAVE)
        (&next[0][0])[k] = 0;
    __syncthreads();
    const int begin = blockIdx.x * CS_BLOCK + wave * CS_STEPS * TPK_WAVE + lane;
    unsigned mine[CS_STEPS];
#pragma unroll
    for (int step = 0; step < CS_STEPS; ++step)
    {
        const int i = begin + step * TPK_WAVE;
        mine[step] = i < n ? keys[i] : ~0u;
        if (i < n)
            atomicAdd(&next[wave][mine[step]], 1u);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < bins; k += CS_WAVES * TPK_WAVE)
    {
        unsigned at = table[(int64_t)k * gridDim.x + blockIdx.x];
        for (int w = 0; w < CS_WAVES; ++w)
        {
            const unsigned c = next[w][k];
            next[w][k] = at;
            at += c;
        }
    }
    __syncthreads();
    // a wavefront's steps follow each other, so its counters need no atomics: the lanes of one key take
    // consecutive places, their last lane moves the counter on
#pragma unroll
    for (int step = 0; step < CS_STEPS; ++step)
    {
        const int i = begin + step * TPK_WAVE;
        const unsigned k = mine[step];
        u64 same = __ballot(i < n);
        for (int bit = 0; bit < bits; ++bit)
        {
            const u64 set = __ballot((k >> bit) & 1u);
            same &= (k >> bit) & 1u ? set : ~set;
        }
        if (i < n)
        {
            const unsigned at = next[wave][k] + tpk_prefix_count(same);
            keys_out[at] = k;
            values_out[at] = (unsigned)i;
        }
        __builtin_amdgcn_wave_barrier();
        if (i < n && (same >> lane) == 1)
            next[wave][k] += __builtin_popcountll(same);
        __builtin_amdgcn_wave_barrier();
    }
}

template <typename Keys>
__global__ void __launch_bounds__(CL_THREADS) sort_keys_kernel(int n, Keys key_of, unsigned* keys, unsigned* values)
{
    const int v = blockIdx.x * CL_THREADS + threadIdx.x;
    if (v >= n)
        return;
    keys[v] = key_of(v);
    values[v] = (unsigned)v;
}

struct SortSpace
{
    unsigned *keys_in, *keys_out, *values_in, *values_out;
    void* temp; // at least CS_TABLE entries
    size_t temp_bytes;
};

// Point numbers 0 .. n-1 sorted by key_of (values below `bins`), equal keys in ascending order.
template <typename Keys>
hipError_t sort_points(int n, unsigned bins, const Keys& key_of, const SortSpace& space, hipStream_t s)
{
    const unsigned bits = bins > 1 ? 32u - (unsigned)__builtin_clz(bins - 1) : 1u;
    const int64_t blocks = tpk_ceil_div(n, CS_BLOCK);
    if (bins <= (unsigned)CS_BINS && blocks * bins <= CS_TABLE)
    {
        unsigned* table = static_cast<unsigned*>(space.temp);
        counting_histogram_kernel<<<(unsigned)blocks, CS_WAVES * TPK_WAVE, 0, s>>>(n, (int)bins, key_of, space.keys_in, table);
        counting_scan_kernel<<<1, CS_SCAN_THREADS, 0, s>>>((int)(blocks * bins), table);
        counting_place_kernel<<<(unsigned)blocks, CS_WAVES * TPK_WAVE, 0, s>>>(n, (int)bins, (int)bits, space.keys_in, table, space.keys_out,
                                                                                space.values_out);
        return hipGetLastError();
    }
    sort_keys_kernel<<<(unsigned)tpk_ceil_div(n, CL_THREADS), CL_THREADS, 0, s>>>(n, key_of, space.keys_in, space.values_in);
    size_t temp_size = space.temp_bytes;
    return rocprim::radix_sort_pairs(space.temp, temp_size, space.keys_in, space.keys_out, space.values_in, space.values_out, (size_t)n,
                                     0u, bits, s);
}

__global__ void __launch_bounds__(CL_THREADS) cluster_widen_kernel(int count, const unsigned* __restrict__ values, int64_t* members)
{
    const int i = blockIdx.x * CL_THREADS + threadIdx.x;
    if (i < count)
        members[i] = values[i];
}

// The reference's walk (cluster.py:15-33), one wavefront per kept cluster: the point taken off
// the stack has its row read by the lanes; the unseen members of the cluster among the entries
// are marked, and appended to the stack and to the cluster in row order.  A member is unseen
// while its label still is the cluster's first point; one compare-and-swap tests and marks it
// (the label becomes the complement), so a point enters once even if a row repeats it, and the
// labels are used up by this kernel.  The stack of a cluster occupies the cluster's own range of
// `stack` (it never holds more than the cluster has members).
__global__ void __launch_bounds__(CL_THREADS)
    cluster_walk_kernel(int n, int nsample, int clusters, const int64_t* __restrict__ neighbours, int* label,
                        const int* __restrict__ seeds, const int64_t* __restrict__ starts, int* stack, int64_t* members)
{
    const int c = blockIdx.x * (CL_THREADS / TPK_WAVE) + threadIdx.x / TPK_WAVE;
    if (c >= clusters)
        return;
    const int lane = (int)tpk_lane_id();
    const int seed = seeds[c];
    const int64_t base = starts[c];
    const int capacity = (int)(starts[c + 1] - base);
    int* my_stack = stack + base;
    int64_t* mine = members + base;
    if (lane == 0)
    {
        label[seed] = ~seed;
        mine[0] = seed;
    }
    int filled = 1, top = 0;
    int k = seed;
    while (true)
    {
        int pushed_last = -1;
        for (int first = 0; first < nsample; first += TPK_WAVE)
        {
            const int j = first + lane;
            const int64_t nei = j < nsample ? neighbours[(int64_t)k * nsample + j] : -1;
            const u64 ends = __ballot(nei == -1);
            const int valid = ends ? __builtin_ctzll(ends) : TPK_WAVE;
            bool take = false;
            if (lane < valid && nei >= 0 && nei < n)
                take = atomicCAS(&label[nei], seed, ~seed) == seed;
            const u64 taken = __ballot(take);
            const int count = __builtin_popcountll(taken);
            if (count > 0 && filled + count <= capacity)
            {
                const int at = (int)tpk_prefix_count(taken);
                if (take)
                {
                    my_stack[top + at] = (int)nei;
                    mine[filled + at] = nei;
                }
                pushed_last = __builtin_amdgcn_readlane((int)nei, 63 - __builtin_clzll(taken));
                top += count;
                filled += count;
            }
            if (ends)
                break;
        }
        if (top == 0)
            break;
        --top;
        if (pushed_last >= 0)
            k = pushed_last;
        else
        {
            __threadfence_block(); // entries written by other lanes in earlier steps
            k = __builtin_amdgcn_readfirstlane(__hip_atomic_load(&my_stack[top], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
        }
    }
}

// ---- pieces for the walk on the host ----------------------------------------------------------

// First parents, and the middle and last valid entry of every row for the two rounds of links below.  Rows
// of an unsorted ball query list ascending indices, so the first entry is the smallest point the row names.
// A parent is never above its point, so chains end.
__global__ void __launch_bounds__(CL_THREADS)
    component_init_kernel(int n, int nsample, const int64_t* __restrict__ neighbours, int* parent, int* picks, int* size, int* largest)
{
    const int64_t t = (int64_t)blockIdx.x * CL_THREADS + threadIdx.x;
    if (t == 0)
        *largest = 0;
    const int64_t point = t / CL_ROW_LANES;
    const int g = (int)(t % CL_ROW_LANES);
    if (point >= n)
        return; // the whole group of lanes leaves together
    const int shift = (int)(tpk_lane_id() & (TPK_WAVE - CL_ROW_LANES)); // first lane of this row's group
    const int64_t* row = neighbours + point * nsample;
    int count = 0;
    for (int first = 0; first < nsample; first += CL_ROW_LANES)
    {
        bool row_ends;
        count += entries_before_end(first + g < nsample ? row[first + g] : -1, shift, &row_ends);
        if (row_ends)
            break;
    }
    const int v = (int)point;
    if (g >= 3)
        return;
    const int64_t nei = count > 0 ? row[g == 0 ? 0 : g == 1 ? count - 1 : count / 2] : -1;
    const bool usable = nei >= 0 && nei < n;
    if (g == 0)
    {
        parent[v] = usable && nei < v ? (int)nei : v;
        size[v] = 0;
    }
    else
        picks[(int64_t)(g - 1) * n + v] = usable ? (int)nei : v;
}

// Joins the trees of two points: the higher root is hung under the lower by compare-and-swap.  The dies'
// L2s do not see each other's stores within a kernel, so a root found by plain reads may have been hung
// meanwhile; it is looked at once more past the caches before the swap is tried, because failing swaps of
// thousands of entries on one address are what this would otherwise spend its time on.  What is found there
// is strictly lower, so the loop ends.
__device__ __forceinline__ void join_trees(int* parent, int a, int b)
{
    a = find_root(parent, a);
    b = find_root(parent, b);
    while (a != b)
    {
        const int high = max(a, b), low = min(a, b);
        int above = __hip_atomic_load(&parent[high], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (above == high)
            above = atomicCAS(&parent[high], high, low);
        if (above == high)
            return;
        a = find_root(parent, above);
        b = low;
    }
}

// One entry of every row.
__global__ void __launch_bounds__(CL_THREADS) component_link_kernel(int n, const int* __restrict__ picks, int* parent)
{
    const int u = blockIdx.x * CL_THREADS + threadIdx.x;
    if (u >= n)
        return;
    const int nei = picks[u];
    if (parent[nei] != parent[u])
        join_trees(parent, u, nei);
}

// Every entry joins the trees of its two points, whatever its direction.  The rounds before have left one
// tree for most of every component and flattened it, so for nearly all entries this is one comparison of
// two parents.
__global__ void __launch_bounds__(CL_THREADS)
    component_join_kernel(int n, int nsample, const int64_t* __restrict__ neighbours, int* parent)
{
    const int64_t t = (int64_t)blockIdx.x * CL_THREADS + threadIdx.x;
    const int64_t point = t / CL_ROW_LANES;
    const int g = (int)(t % CL_ROW_LANES);
    if (point >= n)
        return; // the whole group of lanes leaves together
    const int u = (int)point;
    const int shift = (int)(tpk_lane_id() & (TPK_WAVE - CL_ROW_LANES)); // first lane of this row's group
    const int mine = parent[u];
    for (int first = 0; first < nsample; first += CL_ROW_LANES)
    {
        const int j = first + g;
        const int64_t nei = j < nsample ? neighbours[(int64_t)u * nsample + j] : -1;
        bool row_ends;
        const int valid = entries_before_end(nei, shift, &row_ends);
        if (g < valid && nei >= 0 && nei < n && nei != u && parent[nei] != mine)
            join_trees(parent, u, (int)nei);
        if (row_ends)
            break;
    }
}

// Every point directly under its root (stores of other threads only move a point further up).
__global__ void __launch_bounds__(CL_THREADS) component_flatten_kernel(int n, int* parent)
{
    const int v = blockIdx.x * CL_THREADS + threadIdx.x;
    if (v >= n)
        return;
    const int root = find_root(parent, v);
    if (root < parent[v])
        parent[v] = root;
}

// The root of every point, and the points per root.  Neighbouring points share few roots, so the counts are
// gathered in LDS first (a small open table; what finds no place there is added outside): device-scope atomics
// on one address pass one at a time.
constexpr int CL_ROOT_THREADS = 1024;
constexpr int CL_ROOT_POINTS = 4 * CL_ROOT_THREADS; // per workgroup
constexpr int CL_ROOT_SLOTS = 512;

__global__ void __launch_bounds__(CL_ROOT_THREADS)
    component_roots_kernel(int n, const int* __restrict__ parent, int* __restrict__ root, int* size)
{
    __shared__ int slot_root[CL_ROOT_SLOTS], slot_count[CL_ROOT_SLOTS];
    for (int i = threadIdx.x; i < CL_ROOT_SLOTS; i += CL_ROOT_THREADS)
    {
        slot_root[i] = -1;
        slot_count[i] = 0;
    }
    __syncthreads();
    const int begin = blockIdx.x * CL_ROOT_POINTS + threadIdx.x;
    for (int v = begin; v < n && v < begin + CL_ROOT_POINTS; v += CL_ROOT_THREADS)
    {
        const int r = find_root(parent, v);
        root[v] = r;
        bool counted = false;
        for (int probe = 0; probe < 4 && !counted; ++probe)
        {
            const int slot = (int)((unsigned)r * 0x9E3779B1u >> 23) + probe & (CL_ROOT_SLOTS - 1);
            int holds = slot_root[slot];
            if (holds == -1)
                holds = atomicCAS(&slot_root[slot], -1, r);
            if (holds == -1 || holds == r)
            {
                atomicAdd(&slot_count[slot], 1);
                counted = true;
            }
        }
        if (!counted)
            atomicAdd(&size[r], 1);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < CL_ROOT_SLOTS; i += CL_ROOT_THREADS)
        if (slot_count[i] > 0)
            atomicAdd(&size[slot_root[i]], slot_count[i]);
}

// cluster_kept_kernel's scan input, and the size of the largest piece.
__global__ void __launch_bounds__(CL_THREADS)
    component_kept_kernel(int n, int min_size, const int* __restrict__ root, const int* __restrict__ size, u64* packed, int* largest)
{
    const int v = blockIdx.x * CL_THREADS + threadIdx.x;
    if (v > n)
        return;
    u64 p = 0;
    if (v < n && root[v] == v && size[v] >= min_size)
    {
        p = ((u64)1 << 32) | (unsigned)size[v];
        atomicMax(largest, size[v]);
    }
    packed[v] = p;
}

// info = {pieces, points in them, largest piece}
__global__ void component_info_kernel(int n, const u64* __restrict__ scanned, const int* __restrict__ largest, int64_t* info)
{
    info[0] = (int64_t)(scanned[n] >> 32);
    info[1] = (int64_t)(scanned[n] & 0xffffffffu);
    info[2] = *largest;
}

// Numbers the pieces by size, the largest first: a caller that walks them on host threads has to wait for the end of the longest
// walk, so the rows of the largest piece are the ones it wants first.  number: piece of every root; starts: first place of every piece,
// then the total.  Every thread compares its piece with all others: 5 us for 150 pieces.
constexpr int CL_RANKED = 1024; // pieces at most; more stay in the order of their first points
__global__ void __launch_bounds__(CL_RANKED) component_rank_kernel(int pieces, const int* __restrict__ seeds, int* number, int64_t* starts)
{
    __shared__ int size[CL_RANKED];
    const int i = threadIdx.x;
    const int mine = i < pieces ? (int)(starts[i + 1] - starts[i]) : 0;
    size[i] = mine;
    __syncthreads();
    if (i >= pieces)
        return;
    int rank = 0, at = 0;
    for (int j = 0; j < pieces; ++j)
    {
        const int other = size[j];
        const bool before = other > mine || (other == mine && j < i);
        rank += before ? 1 : 0;
        at += before ? other : 0;
    }
    starts[rank] = at;
    number[seeds[i]] = rank;
}

__global__ void __launch_bounds__(CL_THREADS)
    component_places_kernel(int count, const unsigned* __restrict__ values, int* place, int32_t* positions, int pieces,
                            const int64_t* __restrict__ starts, int64_t* starts_out)
{
    const int i = blockIdx.x * CL_THREADS + threadIdx.x;
    if (i <= pieces) // (a piece has a point at least)
        starts_out[i] = starts[i];
    if (i >= count)
        return;
    const int v = (int)values[i];
    place[v] = i;
    positions[i] = v;
}

// Row i: the entries of the point at place i, as places inside its piece; what lies behind the row's end,
// or outside the matrix, becomes the point itself, which the walk has always seen already - so it needs no
// test for the end of a row.
template <typename E>
__global__ void __launch_bounds__(CL_THREADS)
    component_rows_kernel(int n, int first, int end, int nsample, const int64_t* __restrict__ neighbours, const unsigned* __restrict__ values,
                          const unsigned* __restrict__ keys, const int64_t* __restrict__ starts, const int* __restrict__ place, E* rows)
{
    const int64_t t = (int64_t)blockIdx.x * CL_THREADS + threadIdx.x;
    const int64_t slot = first + t / CL_ROW_LANES;
    const int g = (int)(t % CL_ROW_LANES);
    if (slot >= end)
        return; // the whole group of lanes leaves together
    const int shift = (int)(tpk_lane_id() & (TPK_WAVE - CL_ROW_LANES));
    const int64_t u = values[slot];
    const int base = (int)starts[keys[slot]];
    bool ended = false;
    for (int first = 0; first < nsample; first += CL_ROW_LANES)
    {
        const int j = first + g;
        const int64_t nei = j < nsample ? neighbours[u * nsample + j] : -1;
        bool row_ends;
        const int valid = entries_before_end(nei, shift, &row_ends);
        int entry = (int)slot;
        if (!ended && g < valid && nei >= 0 && nei < n)
            entry = place[nei];
        if (j < nsample)
            rows[slot * nsample + j] = (E)(entry - base);
        ended |= row_ends;
    }
}

// ---- the points of a labelled cloud, label by label ---------------------------------------------

constexpr int RG_RANGE_BLOCKS = 128;

struct Ignored
{
    int count;
    int64_t value[TPK_REGION_IGNORED];
};

struct LabelRange
{
    int64_t low, high, kept;
};

__device__ __forceinline__ bool is_ignored(const Ignored& ignored, int64_t label)
{
    for (int i = 0; i < ignored.count; ++i)
        if (ignored.value[i] == label)
            return true;
    return false;
}

// Smallest and largest label that is not ignored and how many points carry one, per block; behind them the first and the last
// sample id.
__global__ void __launch_bounds__(CL_THREADS)
    region_range_kernel(int n, const int64_t* __restrict__ labels, const int64_t* __restrict__ batch, Ignored ignored, LabelRange* ranges)
{
    __shared__ LabelRange shared[CL_THREADS];
    if (blockIdx.x == 0 && threadIdx.x == 0)
        ranges[RG_RANGE_BLOCKS] = LabelRange{batch[0], batch[n - 1], 0};
    LabelRange r{INT64_MAX, INT64_MIN, 0};
    for (int i = blockIdx.x * CL_THREADS + threadIdx.x; i < n; i += RG_RANGE_BLOCKS * CL_THREADS)
    {
        const int64_t label = labels[i];
        if (is_ignored(ignored, label))
            continue;
        r.low = min(r.low, label);
        r.high = max(r.high, label);
        r.kept += 1;
    }
    shared[threadIdx.x] = r;
    for (int half = CL_THREADS / 2; half > 0; half /= 2)
    {
        __syncthreads();
        if ((int)threadIdx.x < half)
        {
            LabelRange& a = shared[threadIdx.x];
            const LabelRange& b = shared[threadIdx.x + half];
            a.low = min(a.low, b.low);
            a.high = max(a.high, b.high);
            a.kept += b.kept;
        }
    }
    if (threadIdx.x == 0)
        ranges[blockIdx.x] = shared[0];
}

struct RegionKeys
{
    int64_t low;
    unsigned beyond; // key of the points left out
    const int64_t* labels;
    Ignored ignored;
    __device__ __forceinline__ unsigned operator()(int i) const
    {
        const int64_t label = labels[i];
        return is_ignored(ignored, label) ? beyond : (unsigned)(label - low);
    }
};

// Points of one label and one sample form a cloud; its id grows with (label, sample), which is the order
// the rows stand in.  (span: of the sample ids; labels * span is below 2^63, or the caller numbers both anew)
__global__ void __launch_bounds__(CL_THREADS)
    region_gather_kernel(int kept, int64_t first, int64_t span, const unsigned* __restrict__ keys, const unsigned* __restrict__ values,
                         const int64_t* __restrict__ batch, const float* __restrict__ pos, int32_t* order, float* pos_out, int64_t* ids)
{
    const int i = blockIdx.x * CL_THREADS + threadIdx.x;
    if (i >= kept)
        return;
    const int64_t v = values[i];
    order[i] = (int32_t)v;
    ids[i] = (int64_t)keys[i] * span + (batch[v] - first);
    pos_out[(int64_t)i * 3 + 0] = pos[v * 3 + 0];
    pos_out[(int64_t)i * 3 + 1] = pos[v * 3 + 1];
    pos_out[(int64_t)i * 3 + 2] = pos[v * 3 + 2];
}

template <typename P>
__global__ void __launch_bounds__(CL_THREADS)
    region_members_kernel(int64_t count, const int32_t* __restrict__ order, const P* positions, int64_t* members)
{
    const int64_t i = (int64_t)blockIdx.x * CL_THREADS + threadIdx.x;
    if (i >= count)
        return;
    const int64_t p = (int64_t)positions[i];
    members[i] = order ? (int64_t)order[p] : p;
}

// Member i of the clusters, one after the other, as an index: its cluster's row of the table says where the cluster's members lie in members_in
// and from which place its piece's places count.
template <typename E>
__global__ void __launch_bounds__(CL_THREADS)
    grow_members_kernel(int64_t count, int clusters, const int64_t* __restrict__ table, const E* __restrict__ members_in,
                        const int32_t* __restrict__ positions, const int32_t* __restrict__ order, int64_t* members)
{
    const int64_t i = (int64_t)blockIdx.x * CL_THREADS + threadIdx.x;
    if (i >= count)
        return;
    const int c = grow_cluster_of([&](int64_t word) { return table[word]; }, clusters, i);
    const int64_t* cluster = table + GROW_TABLE_ROW * (int64_t)c;
    const int32_t p = positions[cluster[2] + (int64_t)members_in[cluster[1] + (i - cluster[0])]];
    members[i] = order ? (int64_t)order[p] : (int64_t)p;
}

struct Layout
{
    size_t parent, mutual, label, size, number, seeds, stack, keys_in, keys_out, values_in, values_out, packed, scanned, changed,
        temp, temp_bytes, total;
};

// 32-bit words of a point's mask of mutual entries.
int mask_words(int nsample)
{
    return nsample > 0 ? (nsample + 31) / 32 : 1;
}

size_t aligned(size_t v)
{
    return (v + 255) / 256 * 256;
}

// Temporary storage rocPRIM asks for (the larger of the scan's and the sort's); false when it
// cannot say (no device).
bool temp_bytes(int64_t n, size_t* bytes)
{
    size_t scan = 0, sort = 0;
    u64* p64 = nullptr;
    unsigned* p32 = nullptr;
    if (rocprim::exclusive_scan(nullptr, scan, p64, p64, (u64)0, (size_t)n + 1, rocprim::plus<u64>()) != hipSuccess)
        return false;
    if (rocprim::radix_sort_pairs(nullptr, sort, p32, p32, p32, p32, (size_t)n, 0u, 32u) != hipSuccess)
        return false;
    *bytes = scan > sort ? scan : sort;
    if (*bytes < CS_TABLE * sizeof(unsigned))
        *bytes = CS_TABLE * sizeof(unsigned);
    return true;
}

bool layout(int64_t n, int nsample, Layout* l)
{
    size_t temp = 0;
    if (!temp_bytes(n, &temp))
        return false;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t here = at;
        at += aligned(bytes);
        return here;
    };
    const size_t ints = (size_t)n * 4;
    l->parent = take(ints);
    l->mutual = take(ints * (size_t)mask_words(nsample));
    l->label = take(ints);
    l->size = take(ints);
    l->number = take(ints);
    l->seeds = take(ints);
    l->stack = take(ints);
    l->keys_in = take(ints);
    l->keys_out = take(ints);
    l->values_in = take(ints);
    l->values_out = take(ints);
    l->packed = take(((size_t)n + 1) * 8);
    l->scanned = take(((size_t)n + 1) * 8);
    l->changed = take(CL_SWEEPS * 4);
    l->temp = take(temp);
    l->temp_bytes = temp;
    l->total = at;
    return true;
}

struct ComponentLayout
{
    size_t parent, root, size, number, seeds, keys_in, keys_out, values_in, values_out, packed, scanned, starts, largest, info, temp,
        temp_bytes, total;
};

bool component_layout(int64_t n, ComponentLayout* l)
{
    size_t temp = 0;
    if (!temp_bytes(n, &temp))
        return false;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t here = at;
        at += aligned(bytes);
        return here;
    };
    const size_t ints = (size_t)n * 4;
    l->parent = take(ints);
    l->root = take(ints);
    l->size = take(ints);
    l->number = take(ints);
    l->seeds = take(ints);
    l->keys_in = take(ints);
    l->keys_out = take(ints);
    l->values_in = take(ints);
    l->values_out = take(ints);
    l->packed = take(((size_t)n + 1) * 8);
    l->scanned = take(((size_t)n + 1) * 8);
    l->starts = take(((size_t)n + 1) * 8);
    l->largest = take(4);
    l->info = take(24);
    l->temp = take(temp);
    l->temp_bytes = temp;
    l->total = at;
    return true;
}

struct RegionLayout
{
    size_t keys_in, keys_out, values_in, values_out, ranges, temp, temp_bytes, total;
};

bool region_layout(int64_t n, RegionLayout* l)
{
    size_t temp = 0;
    if (!temp_bytes(n, &temp))
        return false;
    const size_t ints = aligned((size_t)n * 4);
    l->keys_in = 0;
    l->keys_out = ints;
    l->values_in = 2 * ints;
    l->values_out = 3 * ints;
    l->ranges = 4 * ints;
    l->temp = l->ranges + aligned((RG_RANGE_BLOCKS + 1) * sizeof(LabelRange));
    l->temp_bytes = temp;
    l->total = l->temp + aligned(temp);
    return true;
}

} // namespace

extern "C" size_t tpk_grow_components_workspace_bytes(int64_t n)
{
    ComponentLayout l;
    if (n <= 0 || n > CL_MAX_POINTS || !component_layout(n, &l))
        return 0;
    return l.total;
}

namespace {

// largest_first: see tpk_grow_components_by_size.
int grow_components(int64_t n, int nsample, const int64_t* neighbours, int64_t min_cluster_size, bool largest_first, int64_t* found,
                    void* workspace, size_t workspace_bytes, void* stream)
{
    if (n <= 0 || nsample <= 0 || !found || !neighbours)
        return TPK_ERR_INVALID_ARG;
    if (n > CL_MAX_POINTS)
        return TPK_ERR_UNSUPPORTED;
    ComponentLayout l;
    if (!component_layout(n, &l))
        return TPK_ERR_UNSUPPORTED;
    if (!workspace || workspace_bytes < l.total || (reinterpret_cast<uintptr_t>(workspace) & 255) != 0)
        return TPK_ERR_WORKSPACE;
    hipStream_t s = tpk_stream(stream);
    char* ws = static_cast<char*>(workspace);
    int* parent = reinterpret_cast<int*>(ws + l.parent);
    int* root = reinterpret_cast<int*>(ws + l.root);
    int* size = reinterpret_cast<int*>(ws + l.size);
    int* number = reinterpret_cast<int*>(ws + l.number);
    unsigned* keys_in = reinterpret_cast<unsigned*>(ws + l.keys_in);
    unsigned* keys_out = reinterpret_cast<unsigned*>(ws + l.keys_out);
    unsigned* values_in = reinterpret_cast<unsigned*>(ws + l.values_in);
    unsigned* values_out = reinterpret_cast<unsigned*>(ws + l.values_out);
    u64* packed = reinterpret_cast<u64*>(ws + l.packed);
    u64* scanned = reinterpret_cast<u64*>(ws + l.scanned);
    int64_t* starts = reinterpret_cast<int64_t*>(ws + l.starts);
    int* largest = reinterpret_cast<int*>(ws + l.largest);
    int64_t* info = reinterpret_cast<int64_t*>(ws + l.info);
    const int ni = (int)n;
    const unsigned blocks = (unsigned)tpk_ceil_div(n, CL_THREADS);
    const unsigned blocks1 = (unsigned)tpk_ceil_div(n + 1, CL_THREADS);
    const unsigned row_blocks = (unsigned)tpk_ceil_div(n * CL_ROW_LANES, CL_THREADS);
    const int min_size = (int)(min_cluster_size > n ? n + 1 : (min_cluster_size < 1 ? 1 : min_cluster_size));
    int* picks = reinterpret_cast<int*>(ws + l.packed); // (2 n ints; the counts come later)
    component_init_kernel<<<row_blocks, CL_THREADS, 0, s>>>(ni, nsample, neighbours, parent, picks, size, largest);
    component_flatten_kernel<<<blocks, CL_THREADS, 0, s>>>(ni, parent);
    for (int round = 0; round < 2; ++round)
    {
        component_link_kernel<<<blocks, CL_THREADS, 0, s>>>(ni, picks + (size_t)round * n, parent);
        component_flatten_kernel<<<blocks, CL_THREADS, 0, s>>>(ni, parent);
    }
    component_join_kernel<<<row_blocks, CL_THREADS, 0, s>>>(ni, nsample, neighbours, parent);
    component_roots_kernel<<<(unsigned)tpk_ceil_div(n, CL_ROOT_POINTS), CL_ROOT_THREADS, 0, s>>>(ni, parent, root, size);
    component_kept_kernel<<<blocks1, CL_THREADS, 0, s>>>(ni, min_size, root, size, packed, largest);
    size_t temp_size = l.temp_bytes;
    hipError_t e = rocprim::exclusive_scan(ws + l.temp, temp_size, packed, scanned, (u64)0, (size_t)n + 1, rocprim::plus<u64>(), s);
    if (e != hipSuccess)
        return (int)e;
    component_info_kernel<<<1, 1, 0, s>>>(ni, scanned, largest, info);
    cluster_describe_kernel<<<blocks1, CL_THREADS, 0, s>>>(ni, packed, scanned, number, reinterpret_cast<int*>(ws + l.seeds), starts);
    e = static_cast<hipError_t>(tpk_read_back(found, info, 24, s));
    if (e != hipSuccess || found[0] == 0)
        return (int)e;
    if (largest_first && found[0] > 1 && found[0] <= CL_RANKED)
        component_rank_kernel<<<1, CL_RANKED, 0, s>>>((int)found[0], reinterpret_cast<const int*>(ws + l.seeds), number, starts);
    e = sort_points(ni, (unsigned)found[0] + 1u, ClusterKeys{(int)found[0], root, number},
                    SortSpace{keys_in, keys_out, values_in, values_out, ws + l.temp, l.temp_bytes}, s);
    return e != hipSuccess ? (int)e : tpk_launch_status();
}

} // namespace

extern "C" int tpk_grow_components(int64_t n, int nsample, const int64_t* neighbours, int64_t min_cluster_size, int64_t* found,
                                   void* workspace, size_t workspace_bytes, void* stream)
{
    return grow_components(n, nsample, neighbours, min_cluster_size, false, found, workspace, workspace_bytes, stream);
}

extern "C" int tpk_grow_components_by_size(int64_t n, int nsample, const int64_t* neighbours, int64_t min_cluster_size, int64_t* found,
                                           void* workspace, size_t workspace_bytes, void* stream)
{
    return grow_components(n, nsample, neighbours, min_cluster_size, true, found, workspace, workspace_bytes, stream);
}

extern "C" int tpk_grow_rows_part(int64_t n, int nsample, const int64_t* neighbours, const int64_t* found, int entry_bytes, int64_t first,
                                  int64_t count, void* rows, void* workspace, size_t workspace_bytes, void* stream)
{
    if (n <= 0 || n > CL_MAX_POINTS || nsample <= 0 || !neighbours || !found || !rows || found[0] < 1 || found[1] < 1 || found[1] > n ||
        (entry_bytes != 2 && entry_bytes != 4) || (entry_bytes == 2 && found[2] > 65536) || first < 0 || count < 0 || first > found[1] - count)
        return TPK_ERR_INVALID_ARG;
    ComponentLayout l;
    if (!component_layout(n, &l))
        return TPK_ERR_UNSUPPORTED;
    if (!workspace || workspace_bytes < l.total || (reinterpret_cast<uintptr_t>(workspace) & 255) != 0)
        return TPK_ERR_WORKSPACE;
    if (count == 0)
        return TPK_OK;
    hipStream_t s = tpk_stream(stream);
    char* ws = static_cast<char*>(workspace);
    const unsigned* keys = reinterpret_cast<const unsigned*>(ws + l.keys_out);
    const unsigned* values = reinterpret_cast<const unsigned*>(ws + l.values_out);
    const int* place = reinterpret_cast<const int*>(ws + l.parent);
    const int64_t* from = reinterpret_cast<const int64_t*>(ws + l.starts);
    const unsigned row_blocks = (unsigned)tpk_ceil_div(count * CL_ROW_LANES, CL_THREADS);
    const int end = (int)(first + count);
    if (entry_bytes == 2)
        component_rows_kernel<uint16_t><<<row_blocks, CL_THREADS, 0, s>>>((int)n, (int)first, end, nsample, neighbours, values, keys, from, place,
                                                                           static_cast<uint16_t*>(rows));
    else
        component_rows_kernel<uint32_t><<<row_blocks, CL_THREADS, 0, s>>>((int)n, (int)first, end, nsample, neighbours, values, keys, from, place,
                                                                           static_cast<uint32_t*>(rows));
    return tpk_launch_status();
}

extern "C" int tpk_grow_places(int64_t n, const int64_t* found, int32_t* positions, int64_t* starts, void* workspace,
                               size_t workspace_bytes, void* stream)
{
    if (n <= 0 || n > CL_MAX_POINTS || !found || !positions || !starts || found[0] < 1 || found[1] < found[0] || found[1] > n)
        return TPK_ERR_INVALID_ARG;
    ComponentLayout l;
    if (!component_layout(n, &l))
        return TPK_ERR_UNSUPPORTED;
    if (!workspace || workspace_bytes < l.total || (reinterpret_cast<uintptr_t>(workspace) & 255) != 0)
        return TPK_ERR_WORKSPACE;
    char* ws = static_cast<char*>(workspace);
    int* place = reinterpret_cast<int*>(ws + l.parent); // (the trees are done with)
    const int count = (int)found[1];
    component_places_kernel<<<(unsigned)tpk_ceil_div((int64_t)count + 1, CL_THREADS), CL_THREADS, 0, tpk_stream(stream)>>>(
        count, reinterpret_cast<const unsigned*>(ws + l.values_out), place, positions, (int)found[0], reinterpret_cast<const int64_t*>(ws + l.starts),
        starts);
    return tpk_launch_status();
}

extern "C" int tpk_grow_rows(int64_t n, int nsample, const int64_t* neighbours, const int64_t* found, int entry_bytes, void* rows,
                             int32_t* positions, int64_t* starts, void* workspace, size_t workspace_bytes, void* stream)
{
    if (nsample <= 0 || !neighbours || !found || !rows || (entry_bytes != 2 && entry_bytes != 4) || (entry_bytes == 2 && found[2] > 65536))
        return TPK_ERR_INVALID_ARG;
    const int status = tpk_grow_places(n, found, positions, starts, workspace, workspace_bytes, stream);
    return status != TPK_OK
               ? status
               : tpk_grow_rows_part(n, nsample, neighbours, found, entry_bytes, 0, found[1], rows, workspace, workspace_bytes, stream);
}

extern "C" size_t tpk_region_order_workspace_bytes(int64_t n)
{
    RegionLayout l;
    if (n <= 0 || n > CL_MAX_POINTS || !region_layout(n, &l))
        return 0;
    return l.total;
}

extern "C" int tpk_region_order(int64_t n, const int64_t* labels, const int64_t* batch, const float* pos, int ignored_count,
                                const int64_t* ignored_labels, int64_t* found, int32_t* order, float* pos_out, int64_t* ids,
                                void* workspace, size_t workspace_bytes, void* stream)
{
    if (n <= 0 || !labels || !batch || !pos || !found || !order || !pos_out || !ids || ignored_count < 0 ||
        ignored_count > TPK_REGION_IGNORED || (ignored_count > 0 && !ignored_labels))
        return TPK_ERR_INVALID_ARG;
    if (n > CL_MAX_POINTS)
        return TPK_ERR_UNSUPPORTED;
    RegionLayout l;
    if (!region_layout(n, &l))
        return TPK_ERR_UNSUPPORTED;
    if (!workspace || workspace_bytes < l.total || (reinterpret_cast<uintptr_t>(workspace) & 255) != 0)
        return TPK_ERR_WORKSPACE;
    hipStream_t s = tpk_stream(stream);
    char* ws = static_cast<char*>(workspace);
    Ignored ignored{};
    ignored.count = ignored_count;
    for (int i = 0; i < ignored_count; ++i)
        ignored.value[i] = ignored_labels[i];
    LabelRange* ranges = reinterpret_cast<LabelRange*>(ws + l.ranges);
    region_range_kernel<<<RG_RANGE_BLOCKS, CL_THREADS, 0, s>>>((int)n, labels, batch, ignored, ranges);
    LabelRange host[RG_RANGE_BLOCKS + 1], all{INT64_MAX, INT64_MIN, 0};
    hipError_t e = static_cast<hipError_t>(tpk_read_back(host, ranges, sizeof(host), s));
    if (e != hipSuccess)
        return (int)e;
    for (int block = 0; block < RG_RANGE_BLOCKS; ++block)
    {
        const LabelRange& r = host[block];
        all.low = r.low < all.low ? r.low : all.low;
        all.high = r.high > all.high ? r.high : all.high;
        all.kept += r.kept;
    }
    found[0] = all.kept;
    found[1] = 0;
    if (all.kept == 0)
        return TPK_OK;
    if (all.low == all.high && all.kept == n)
        return TPK_OK; // one label: the points stand in their order already
    if ((uint64_t)all.high - (uint64_t)all.low >= (uint64_t)0x7fffffff)
        return TPK_ERR_UNSUPPORTED;
    const unsigned beyond = (unsigned)(all.high - all.low) + 1u;
    const int64_t first = host[RG_RANGE_BLOCKS].low;
    const uint64_t span = (uint64_t)host[RG_RANGE_BLOCKS].high - (uint64_t)first + 1; // (0: all of them)
    if (!region_ids_fit(beyond, span))
        return TPK_ERR_UNSUPPORTED;
    unsigned* keys_in = reinterpret_cast<unsigned*>(ws + l.keys_in);
    unsigned* keys_out = reinterpret_cast<unsigned*>(ws + l.keys_out);
    unsigned* values_in = reinterpret_cast<unsigned*>(ws + l.values_in);
    unsigned* values_out = reinterpret_cast<unsigned*>(ws + l.values_out);
    e = sort_points((int)n, beyond + 1u, RegionKeys{all.low, beyond, labels, ignored},
                    SortSpace{keys_in, keys_out, values_in, values_out, ws + l.temp, l.temp_bytes}, s);
    if (e != hipSuccess)
        return (int)e;
    region_gather_kernel<<<(unsigned)tpk_ceil_div(all.kept, CL_THREADS), CL_THREADS, 0, s>>>((int)all.kept, first, (int64_t)span, keys_out,
                                                                                             values_out, batch, pos, order, pos_out, ids);
    found[1] = 1;
    return tpk_launch_status();
}

extern "C" int tpk_region_members(int64_t count, const int32_t* order, int position_bytes, const void* positions, int64_t* members,
                                  void* stream)
{
    if (count < 0 || (position_bytes != 4 && position_bytes != 8))
        return TPK_ERR_INVALID_ARG;
    if (count == 0)
        return TPK_OK;
    if (!positions || !members)
        return TPK_ERR_INVALID_ARG;
    const unsigned blocks = (unsigned)tpk_ceil_div(count, CL_THREADS);
    if (position_bytes == 4)
        region_members_kernel<int32_t><<<blocks, CL_THREADS, 0, tpk_stream(stream)>>>(count, order, static_cast<const int32_t*>(positions), members);
    else
        region_members_kernel<int64_t><<<blocks, CL_THREADS, 0, tpk_stream(stream)>>>(count, order, static_cast<const int64_t*>(positions), members);
    return tpk_launch_status();
}

extern "C" int tpk_grow_members(int64_t count, int64_t clusters, const int64_t* table, int entry_bytes, const void* entries,
                                const int32_t* positions, const int32_t* order, int64_t* members, void* stream)
{
    if (count < 0 || clusters < 0 || clusters > CL_MAX_POINTS || (entry_bytes != 2 && entry_bytes != 4))
        return TPK_ERR_INVALID_ARG;
    if (count == 0 || clusters == 0)
        return TPK_OK;
    if (!table || !entries || !positions || !members)
        return TPK_ERR_INVALID_ARG;
    const unsigned blocks = (unsigned)tpk_ceil_div(count, CL_THREADS);
    if (entry_bytes == 2)
        grow_members_kernel<<<blocks, CL_THREADS, 0, tpk_stream(stream)>>>(count, (int)clusters, table, static_cast<const uint16_t*>(entries),
                                                                           positions, order, members);
    else
        grow_members_kernel<<<blocks, CL_THREADS, 0, tpk_stream(stream)>>>(count, (int)clusters, table, static_cast<const uint32_t*>(entries),
                                                                           positions, order, members);
    return tpk_launch_status();
}

extern "C" size_t tpk_grow_proximity_workspace_bytes(int64_t n, int nsample)
{
    Layout l;
    if (n <= 0 || n > CL_MAX_POINTS || nsample < 0 || !layout(n, nsample, &l))
        return 0;
    return l.total;
}

extern "C" int tpk_grow_proximity(int64_t n, int nsample, const int64_t* neighbours, int64_t min_cluster_size,
                                  int member_order, int64_t* members, int64_t* starts, int64_t* found,
                                  void* workspace, size_t workspace_bytes, void* stream)
{
    if (n < 0 || nsample < 0 || !found || (member_order != TPK_MEMBERS_AS_REFERENCE && member_order != TPK_MEMBERS_BY_INDEX))
        return TPK_ERR_INVALID_ARG;
    found[0] = found[1] = 0;
    if (n == 0)
        return TPK_OK;
    if (!members || !starts || (nsample > 0 && !neighbours))
        return TPK_ERR_INVALID_ARG;
    if (n > CL_MAX_POINTS)
        return TPK_ERR_UNSUPPORTED;
    Layout l;
    if (!layout(n, nsample, &l))
        return TPK_ERR_UNSUPPORTED;
    if (!workspace || workspace_bytes < l.total || (reinterpret_cast<uintptr_t>(workspace) & 255) != 0)
        return TPK_ERR_WORKSPACE;
    hipStream_t s = tpk_stream(stream);
    char* ws = static_cast<char*>(workspace);
    int* parent = reinterpret_cast<int*>(ws + l.parent);
    unsigned* mutual = reinterpret_cast<unsigned*>(ws + l.mutual);
    int* label = reinterpret_cast<int*>(ws + l.label);
    int* size = reinterpret_cast<int*>(ws + l.size);
    int* number = reinterpret_cast<int*>(ws + l.number);
    int* seeds = reinterpret_cast<int*>(ws + l.seeds);
    int* stack = reinterpret_cast<int*>(ws + l.stack);
    unsigned* keys_in = reinterpret_cast<unsigned*>(ws + l.keys_in);
    unsigned* keys_out = reinterpret_cast<unsigned*>(ws + l.keys_out);
    unsigned* values_in = reinterpret_cast<unsigned*>(ws + l.values_in);
    unsigned* values_out = reinterpret_cast<unsigned*>(ws + l.values_out);
    u64* packed = reinterpret_cast<u64*>(ws + l.packed);
    u64* scanned = reinterpret_cast<u64*>(ws + l.scanned);
    int* changed = reinterpret_cast<int*>(ws + l.changed);
    void* temp = ws + l.temp;
    size_t temp_size = l.temp_bytes;

    const int ni = (int)n;
    const unsigned blocks = (unsigned)tpk_ceil_div(n, CL_THREADS);
    const unsigned blocks1 = (unsigned)tpk_ceil_div(n + 1, CL_THREADS);
    const unsigned sweep_blocks = (unsigned)tpk_ceil_div(n * CL_ROW_LANES, CL_THREADS);
    const int min_size = (int)(min_cluster_size > n ? n + 1 : (min_cluster_size < 0 ? 0 : min_cluster_size));

    const int words = mask_words(nsample);
    // `stack` serves the sweeps as `handed` first
    cluster_init_kernel<<<blocks, CL_THREADS, 0, s>>>(ni, words, parent, label, size, stack, mutual, changed);
    if (nsample > 0)
    {
        // Enqueues batches of sweeps until the last sweep of a batch reports no change.
        auto until_stable = [&](auto&& launch) -> hipError_t {
            while (true)
            {
                for (int sweep = 0; sweep < CL_SWEEPS; ++sweep)
                    launch(sweep);
                int last = 0;
                const hipError_t e = static_cast<hipError_t>(tpk_read_back(&last, changed + CL_SWEEPS - 1, sizeof(int), s));
                cluster_clear_kernel<<<1, CL_THREADS, 0, s>>>(changed);
                if (e != hipSuccess || last == 0)
                    return e;
            }
        };
        cluster_mutual_kernel<<<sweep_blocks, CL_THREADS, 0, s>>>(ni, nsample, words, neighbours, mutual, parent);
        hipError_t e = until_stable([&](int sweep) {
            cluster_jump_kernel<<<blocks, CL_THREADS, 0, s>>>(ni, parent, changed, sweep);
            cluster_merge_kernel<<<sweep_blocks, CL_THREADS, 0, s>>>(ni, nsample, words, neighbours, mutual, parent, changed, sweep);
        });
        if (e != hipSuccess)
            return (int)e;
        cluster_flatten_kernel<<<blocks, CL_THREADS, 0, s>>>(ni, parent);
        e = until_stable([&](int sweep) {
            cluster_sweep_kernel<<<sweep_blocks, CL_THREADS, 0, s>>>(ni, nsample, neighbours, parent, label, stack, changed, sweep);
        });
        if (e != hipSuccess)
            return (int)e;
        cluster_spread_kernel<<<blocks, CL_THREADS, 0, s>>>(ni, parent, label);
    }
    cluster_count_kernel<<<blocks, CL_THREADS, 0, s>>>(ni, label, size);
    cluster_kept_kernel<<<blocks1, CL_THREADS, 0, s>>>(ni, min_size, label, size, packed);
    hipError_t e = rocprim::exclusive_scan(temp, temp_size, packed, scanned, (u64)0, (size_t)n + 1, rocprim::plus<u64>(), s);
    if (e != hipSuccess)
        return (int)e;
    cluster_describe_kernel<<<blocks1, CL_THREADS, 0, s>>>(ni, packed, scanned, number, seeds, starts);
    u64 totals = 0;
    e = static_cast<hipError_t>(tpk_read_back(&totals, scanned + n, sizeof(u64), s));
    if (e != hipSuccess)
        return (int)e;
    const int clusters = (int)(totals >> 32);
    const int kept_points = (int)(totals & 0xffffffffu);
    found[0] = clusters;
    found[1] = kept_points;
    if (clusters == 0)
        return tpk_launch_status();
    if (member_order == TPK_MEMBERS_BY_INDEX)
    {
        e = sort_points(ni, (unsigned)clusters + 1u, ClusterKeys{clusters, label, number},
                        SortSpace{keys_in, keys_out, values_in, values_out, temp, l.temp_bytes}, s);
        if (e != hipSuccess)
            return (int)e;
        cluster_widen_kernel<<<(unsigned)tpk_ceil_div(kept_points, CL_THREADS), CL_THREADS, 0, s>>>(kept_points, values_out, members);
    }
    else
    {
        const int per_block = CL_THREADS / TPK_WAVE;
        cluster_walk_kernel<<<(unsigned)tpk_ceil_div(clusters, per_block), CL_THREADS, 0, s>>>(
            ni, nsample, clusters, neighbours, label, seeds, starts, stack, members);
    }
    return tpk_launch_status();
}
