// k nearest neighbours, dense layout: for every query point the k nearest support points of the
// same cloud, ascending by (squared distance, index).
//
// The reference offers this operator on the CPU only (torch_points_kernels/knn.py:4-18 raises for
// CUDA tensors; cpu/src/knn.cpp:8-59 runs nanoflann per cloud).  Semantics here: squared fp32
// distances evaluated like three_nn's; equal distances keep the lower index first, as the
// reference's three_nn kernel does (cuda/src/interpolate_gpu.cu:9-65) - nanoflann's order among
// exactly equal distances is unspecified.  k must not exceed the number of support points
// (cpu/src/knn.cpp:12-14 raises).
//
// Up to KNC_MAX_K neighbours are found by a wavefront per query (survivors.h), over a grid in memory up to KNQ_MAX_K of many queries by a
// quarter of one: in clouds that fit into LDS over a grid there (below), in larger ones, given a workspace, over such a grid in memory.  More neighbours, and large clouds without a
// workspace: one lane owns one query and keeps its list in registers (topk.h), 32 entries a round - over
// curve-ordered cells for clouds of 512..163840 points with a workspace, otherwise testing all pairs: the support points of
// the cloud stream through LDS in tiles of float4, read by all lanes at the same address.
#include "ball_cells.h"
#include "lds_grid.h"
#include "nn_grid.h"
#include "survivors.h"
#include "topk.h"

#include <algorithm>
#include <cmath>

namespace {

constexpr int KNN_THREADS = 256;
constexpr int KNN_TILE = 1024; // support points per LDS tile (16 KiB)

constexpr int KNG_AXIS = 128; // cells per axis of a grid in memory at most (LG_AXIS of one in LDS)

constexpr int KNN_GROUP = 8;   // candidates whose distances are formed together

// The `cnt` candidates of an LDS tile (indices base, base + 1, ...) offered to the lane's list.
// Distances are formed KNN_GROUP at a time, so that the LDS reads overlap; the list is only
// touched when the nearest of a group can enter it.
template <int K>
__device__ __forceinline__ void scan_tile(const float4* tile, int cnt, int base, float qx, float qy, float qz,
                                          NearestK<K>& s)
{
    float worst = s.worst();
    int c = 0;
    for (; c + KNN_GROUP <= cnt; c += KNN_GROUP)
    {
        float d[KNN_GROUP];
        float nearest = 0.f;
#pragma unroll
        for (int i = 0; i < KNN_GROUP; ++i)
        {
            const float4 p = tile[c + i];
            d[i] = tpk_dist2(qx, qy, qz, p.x, p.y, p.z);
            nearest = i == 0 ? d[i] : fminf(nearest, d[i]);
        }
        if (nearest <= worst)
        {
#pragma unroll
            for (int i = 0; i < KNN_GROUP; ++i)
            {
                const unsigned long long cand = knn_key(d[i], base + c + i);
                if (s.admits(cand))
                    s.insert(cand);
            }
            worst = s.worst();
        }
    }
    for (; c < cnt; ++c)
    {
        const float4 p = tile[c];
        const unsigned long long cand = knn_key(tpk_dist2(qx, qy, qz, p.x, p.y, p.z), base + c);
        if (s.admits(cand))
            s.insert(cand);
    }
}

// first: number of entries found by earlier rounds; count: entries this round finds (<= K).
template <int K>
__global__ __launch_bounds__(KNN_THREADS) void knn_kernel(
    int n, int m, int k, int first, int count, float limit, int blocks_per_cloud, const float* __restrict__ query,
    const float* __restrict__ support, float* __restrict__ dist2, int64_t* __restrict__ idx)
{
    __shared__ float4 tile[KNN_TILE];

    const int cloud = blockIdx.x / blocks_per_cloud;
    const int blk = blockIdx.x - cloud * blocks_per_cloud;
    query += static_cast<int64_t>(cloud) * n * 3;
    support += static_cast<int64_t>(cloud) * m * 3;
    dist2 += static_cast<int64_t>(cloud) * n * k;
    idx += static_cast<int64_t>(cloud) * n * k;

    const int tid = threadIdx.x;
    const int j = blk * KNN_THREADS + tid;
    const bool real = j < n;
    const int jj = real ? j : n - 1; // lanes past the end shadow the last query and store nothing
    const float qx = query[jj * 3 + 0], qy = query[jj * 3 + 1], qz = query[jj * 3 + 2];
    NearestK<K> s;
    {
        // the last pair of the round before (rounds of one call run one after the other)
        const int64_t at = static_cast<int64_t>(jj) * k + first - 1;
        s.reset(first > 0, first > 0 ? dist2[at] : 0.f, first > 0 ? static_cast<int>(idx[at]) : 0, !real, limit);
    }

    for (int base = 0; base < m; base += KNN_TILE)
    {
        const int cnt = min(KNN_TILE, m - base);
        __syncthreads(); // the previous tile has been consumed by every wave
        for (int t = tid; t < KNN_TILE; t += KNN_THREADS)
        {
            float4 p;
            if (t < cnt)
            {
                const float* src = support + static_cast<int64_t>(base + t) * 3;
                p = make_float4(src[0], src[1], src[2], 0.f);
            }
            else
            {
                // Padding: infinitely far away, with an index no list admits.
                p = make_float4(__builtin_inff(), __builtin_inff(), __builtin_inff(), 0.f);
            }
            tile[t] = p;
        }
        __syncthreads();

        scan_tile<K>(tile, cnt, base, qx, qy, qz, s);
    }

    if (real)
    {
#pragma unroll
        for (int e = 0; e < K; ++e)
            if (e < count)
            {
                dist2[static_cast<int64_t>(j) * k + first + e] = s.dist(e);
                idx[static_cast<int64_t>(j) * k + first + e] = s.index(e);
            }
    }
}

template <int K>
int launch_knn(int b, int n, int m, int k, float limit, const float* query, const float* support, float* dist2,
               int64_t* idx, hipStream_t stream)
{
    const int64_t blocks_per_cloud = tpk_ceil_div(n, KNN_THREADS);
    const int64_t blocks = blocks_per_cloud * b;
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    for (int first = 0; first < k; first += K)
    {
        hipLaunchKernelGGL(knn_kernel<K>, dim3(static_cast<unsigned>(blocks)), dim3(KNN_THREADS), 0, stream, n, m,
                           k, first, k - first < K ? k - first : K, limit, static_cast<int>(blocks_per_cloud), query,
                           support, dist2, idx);
        const int st = tpk_launch_status();
        if (st != TPK_OK)
            return st;
    }
    return TPK_OK;
}

// Distance along axis a from a query (at t, in cells) to cell `at`, a lower bound.
template <bool MEMORY>
__device__ __forceinline__ float cell_apart(const LdsGrid& grid, const float* t, int a, int at)
{
    float near_end = static_cast<float>(at), far_end = static_cast<float>(at + 1);
    if constexpr (MEMORY) // (its outermost cells hold all points that lie beyond them)
    {
        near_end = at == 0 ? grid.below[a] : near_end;
        far_end = at == grid.cells[a] - 1 ? grid.above[a] : far_end;
    }
    const float gap = fmaxf(near_end - t[a], t[a] - far_end);
    return fmaxf(gap - 1e-5f * (fabsf(t[a]) + static_cast<float>(KNG_AXIS)), 0.0f) * grid.width[a];
}

// The cells of row (y, z) within the ball of squared radius `bound` around the query: of what is left of the radius in this row (for a
// query far from the cloud the ball is much wider than the stretch of a row that it reaches).  False: none.
template <bool MEMORY>
__device__ __forceinline__ bool ball_row(const LdsGrid& grid, const float* t, float bound, int y, int z, int& x_from, int& x_to)
{
    const float dy = cell_apart<MEMORY>(grid, t, 1, y), dz = cell_apart<MEMORY>(grid, t, 2, z);
    const float rest = bound * 1.00001f - (dy * dy + dz * dz);
    const float span = __builtin_amdgcn_sqrtf(fmaxf(rest, 0.0f)) * 1.00001f * grid.inv[0] + 1e-5f * (fabsf(t[0]) + static_cast<float>(KNG_AXIS));
    x_from = lg_cell(t[0] - span, grid.cells[0]), x_to = lg_cell(t[0] + span, grid.cells[0]);
    return rest >= 0.0f;
}

// Narrows the rows from[1 .. 2] to to[1 .. 2] of the ball around a query more than a cell outside the cloud to what the cloud's distance
// along the other axes leaves of the ball's radius (a row's cells are trimmed by ball_row).  False: a query not so far out.
__device__ __forceinline__ bool ball_rows_of_far_query(const LdsGrid& grid, const float* t, float bound, int* from, int* to)
{
    float gap[3]; // from the query to the cloud, in cells
#pragma unroll
    for (int a = 0; a < 3; ++a)
        gap[a] = fmaxf(grid.below[a] - t[a], t[a] - grid.above[a]);
    if (!(fmaxf(fmaxf(gap[0], gap[1]), gap[2]) > 1.0f))
        return false;
    float out[3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
    {
        const float apart = fmaxf(gap[a] - 1e-5f * (fabsf(t[a]) + static_cast<float>(KNG_AXIS)), 0.0f) * grid.width[a];
        out[a] = apart * apart;
    }
#pragma unroll
    for (int a = 1; a < 3; ++a)
    {
        const float left = __builtin_amdgcn_sqrtf(fmaxf(bound * 1.00001f - (out[0] + out[3 - a]), 0.0f)) * 1.00001f;
        const float span = left * grid.inv[a] + 1e-5f * (fabsf(t[a]) + static_cast<float>(KNG_AXIS));
        from[a] = lg_cell(t[a] - span, grid.cells[a]);
        to[a] = lg_cell(t[a] + span, grid.cells[a]);
    }
    return true;
}

// One query by one wavefront over a grid of cells: the 27 cells around it hold k points or the block grows; the k-th of
// them bounds the ball the answer lies in, and the cells that ball touches outside the block are examined too (one query
// in three).  The lanes find the candidates of the wavefront's rows of cells by a running maximum: each row's lane leaves
// its number at its first candidate's place.  Returns the lane's key of the answer and its place there (>= k: none).
// m: records in `points`, for the queries no distance separates.  MEMORY: a grid in memory, where a query far from the cloud or with
// hardly any point near it has more cells to pass over than the steps that avoid them cost (in LDS, at most 16 x 16 rows: 0.8 us a
// call for every caller).
template <bool MEMORY>
__device__ __forceinline__ int nearest_in_grid(const LdsGrid& grid, const float4* points, const int* starts, int m, int k, int lane, float qx,
                                                    float qy, float qz, Survivors& s, u64& mine TPK_WORK_PARAM)
{
    const int cx = grid.cells[0], cy = grid.cells[1], cz = grid.cells[2];
    const float q[3] = {qx, qy, qz};
    s.clear();
    s.unit = 0.0f;
    bool separated = true; // every selection so far found its distance

    // The candidates of up to 64 rows of cells, a row per lane (start, size), offered.
    auto walk = [&](int start, int size, int before, int total) __attribute__((always_inline)) {
        const int origin = start - before; // candidate c of the walk lies at origin + c, for the c of this lane's row
        for (int c0 = 0; c0 < total && separated; c0 += TPK_WAVE)
        {
            // the row of candidate c0, and every row that starts behind it in this step at its first candidate
            const int first = __builtin_ctzll(__ballot(size > 0 && before <= c0 && before + size > c0));
            const bool starts_here = size > 0 && before > c0 && before < c0 + TPK_WAVE;
            const int mark = __builtin_amdgcn_ds_permute((starts_here ? before - c0 : 0) << 2, starts_here ? lane : 0);
            const int row = max(wave_inclusive_max_i32(lane == 0 ? 0 : mark), first);
            const int at = __shfl(origin, row) + c0 + lane;
            const bool has = c0 + lane < total;
            const float4 p = points[has ? at : 0];
            TPK_WORK_ADD(1);
            separated = s.offer(has, tpk_dist2(qx, qy, qz, p.x, p.y, p.z), __float_as_int(p.w));
        }
    };

    // ---- the block of cells around the query that holds k points ----
    int c[3];
    float t[3]; // in cells
    for (int a = 0; a < 3; ++a)
    {
        t[a] = (q[a] - grid.lo[a]) * grid.inv[a];
        c[a] = __builtin_amdgcn_readfirstlane(lg_cell(t[a], grid.cells[a]));
    }
    int xl, xh, yl, yh, zl, zh;
    // (a crowded cell may do alone: its 26 neighbours would be as crowded)
    const int own = c[0] + cx * (c[1] + cy * c[2]);
    for (int ring = starts[own + 1] - starts[own] >= 2 * k ? 0 : 1;; ring = ring < 3 ? ring + 1 : MEMORY ? 2 * ring : LG_AXIS)
    {
        xl = max(c[0] - ring, 0), xh = min(c[0] + ring, cx - 1);
        yl = max(c[1] - ring, 0), yh = min(c[1] + ring, cy - 1);
        zl = max(c[2] - ring, 0), zh = min(c[2] + ring, cz - 1);
        const int ny = yh - yl + 1, rows = ny * (zh - zl + 1);
        if (ring <= 3) // (7 x 7 rows are the most a lane each can take)
        {
            int start = 0, size = 0;
            if (lane < rows)
            {
                const int iz = static_cast<int>((static_cast<float>(lane) + 0.5f) * __builtin_amdgcn_rcpf(static_cast<float>(ny)));
                const int c0 = xl + cx * ((yl + lane - iz * ny) + cy * (zl + iz));
                start = starts[c0];
                size = starts[c0 + (xh - xl + 1)] - start;
            }
            const int before = wave_exclusive_sum(size);
            const int total = __builtin_amdgcn_readlane(before + size, TPK_WAVE - 1);
            if (total < k)
                continue;
            // a ball that holds one of them, of the block's volume: 3 / (4 pi) x cells / total
            s.unit = s.volume_ratio(0.2387f * grid.volume * static_cast<float>(rows * (xh - xl + 1)) * __builtin_amdgcn_rcpf(static_cast<float>(total)));
            walk(start, size, before, total);
            break;
        }
        // A query with hardly any point near it: the block doubled until it holds k, over as many steps as its rows take.  (All rows
        // at once: 100000 points of a normal distribution, 4096 queries of them, k = 16: 658 us, this way 124.)
        int total = MEMORY ? 0 : m;
        if constexpr (MEMORY)
        {
            for (int row = lane; row - lane < rows; row += TPK_WAVE)
                if (row < rows)
                {
                    const int iz = static_cast<int>((static_cast<float>(row) + 0.5f) * __builtin_amdgcn_rcpf(static_cast<float>(ny)));
                    const int c0 = xl + cx * ((yl + row - iz * ny) + cy * (zl + iz));
                    total += starts[c0 + (xh - xl + 1)] - starts[c0];
                }
            total = __builtin_amdgcn_readlane(wave_exclusive_sum(total) + total, TPK_WAVE - 1);
            if (total < k && rows * (xh - xl + 1) < cx * cy * cz)
                continue;
        }
        s.unit = s.volume_ratio(0.2387f * grid.volume * static_cast<float>(rows * (xh - xl + 1)) * __builtin_amdgcn_rcpf(static_cast<float>(total)));
        for (int row0 = 0; row0 < rows && separated; row0 += TPK_WAVE)
        {
            const int row = min(row0 + lane, rows - 1);
            const int iz = static_cast<int>((static_cast<float>(row) + 0.5f) * __builtin_amdgcn_rcpf(static_cast<float>(ny)));
            const int c0 = xl + cx * ((yl + row - iz * ny) + cy * (zl + iz));
            const int start = starts[c0], size = row0 + lane < rows ? starts[c0 + (xh - xl + 1)] - start : 0;
            const int before = wave_exclusive_sum(size);
            walk(start, size, before, __builtin_amdgcn_readlane(before + size, TPK_WAVE - 1));
        }
        break;
    }

    // ---- the k-th so far bounds the ball; the cells it touches outside the block ----
    mine = ~0ull;
    int place = KNC_MOST;
    separated = separated && s.count >= k && (s.count <= KNC_MOST || s.select(__builtin_inff(), 0));
    if (separated)
    {
        place = s.rank(mine);
        const int kth = __builtin_ctzll(__ballot(place == k - 1));
        const float bound = tpk_read_lane(__int_as_float(static_cast<int>(mine >> 32)), kth);
        const float radius = __builtin_amdgcn_sqrtf(bound) * 1.00001f;
        int from[3], to[3];
        for (int a = 0; a < 3; ++a)
        {
            // (the ends further out than rounding may have moved a point's cell by)
            const float span = radius * grid.inv[a] + 1e-5f * (fabsf(t[a]) + static_cast<float>(KNG_AXIS));
            from[a] = __builtin_amdgcn_readfirstlane(lg_cell(t[a] - span, grid.cells[a]));
            to[a] = __builtin_amdgcn_readfirstlane(lg_cell(t[a] + span, grid.cells[a]));
        }
        if (from[0] < xl || to[0] > xh || from[1] < yl || to[1] > yh || from[2] < zl || to[2] > zh)
        {
            if constexpr (MEMORY)
            {
                if (ball_rows_of_far_query(grid, t, bound, from, to))
                    for (int a = 1; a < 3; ++a)
                    {
                        from[a] = __builtin_amdgcn_readfirstlane(from[a]);
                        to[a] = __builtin_amdgcn_readfirstlane(to[a]);
                    }
            }
            // the k kept in order, then the rest of the ball: two pieces for a row that crosses the block
            if (place < k)
                s.keys[place] = mine;
            s.count = k;
            s.reach = bound;
            const int ny = to[1] - from[1] + 1, pieces = 2 * ny * (to[2] - from[2] + 1);
            for (int piece0 = 0; piece0 < pieces && separated; piece0 += TPK_WAVE)
            {
                const int e = piece0 + lane;
                int start = 0, size = 0;
                if (e < pieces)
                {
                    const bool right = e & 1;
                    const int row = e >> 1;
                    const int iz = static_cast<int>((static_cast<float>(row) + 0.5f) * __builtin_amdgcn_rcpf(static_cast<float>(ny)));
                    const int y = from[1] + row - iz * ny, z = from[2] + iz;
                    const bool crosses = y >= yl && y <= yh && z >= zl && z <= zh;
                    int x_from, x_to;
                    const bool touched = ball_row<MEMORY>(grid, t, bound, y, z, x_from, x_to);
                    const int x0 = right ? max(xh + 1, x_from) : x_from;
                    const int x1 = right ? (crosses ? x_to : -1) : (crosses ? min(xl - 1, x_to) : x_to);
                    if (touched && x1 >= x0)
                    {
                        const int c0 = cx * (y + cy * z);
                        start = starts[c0 + x0];
                        size = starts[c0 + x1 + 1] - start;
                    }
                }
                const int before = wave_exclusive_sum(size);
                walk(start, size, before, __builtin_amdgcn_readlane(before + size, TPK_WAVE - 1));
            }
            separated = separated && (s.count <= KNC_MOST || s.select(__builtin_inff(), 0));
            if (separated && (s.count > k || s.reach != bound)) // (else none came along, and the k lie in order)
                place = s.rank(mine);
            else if (separated)
                place = lane < k ? lane : KNC_MOST, mine = s.keys[lane < k ? lane : 0];
        }
    }
    if (!separated)
    {
        mine = nearest_by_merging(m, k, lane, qx, qy, qz, [&](int at) { return points[at]; } TPK_WORK_ARG);
        place = lane;
    }
    return place;
}

// Points per cell: a fifth of k, so that the 27 cells around a query hold five times k and the ball inside them rather more
// than k.  (0.15 and 0.32 of k: within 4 % on even clouds; on a sphere 0.32 is 8 to 12 % slower.)
inline float knn_per_cell(int k)
{
    return fmaxf(1.0f, 0.2f * static_cast<float>(k));
}

// Clouds of up to LG_MAX_POINTS points: every workgroup builds the grid in LDS (lds_grid.h) and serves a stretch of queries.
__global__ __launch_bounds__(LG_THREADS) void knn_cells_kernel(
    int n, int m, int k, int blocks_per_cloud, int queries_per_block, float per_cell, const float* __restrict__ query,
    const float* __restrict__ support, float* __restrict__ dist2, int64_t* __restrict__ idx)
{
    extern __shared__ __align__(16) unsigned char knc_lds[];
    const int tid = threadIdx.x;
    const int lane = tid & (TPK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / TPK_WAVE);
    const int cloud = blockIdx.x / blocks_per_cloud;
    const int blk = blockIdx.x - cloud * blocks_per_cloud;
    query += static_cast<int64_t>(cloud) * n * 3;
    support += static_cast<int64_t>(cloud) * m * 3;
    dist2 += static_cast<int64_t>(cloud) * n * k;
    idx += static_cast<int64_t>(cloud) * n * k;
    TPK_WORK_DECL

    u64* const all_keys = reinterpret_cast<u64*>(knc_lds);
    LdsGrid grid;
    lds_grid_build(grid, knc_lds + LG_WAVES * KNC_ROOM * sizeof(u64), support, m, 0, per_cell);
    Survivors s;
    s.keys = all_keys + wave * KNC_ROOM;
    s.lane = lane;
    s.k = k;

    const int q_end = min(n, (blk + 1) * queries_per_block);
    for (int j = blk * queries_per_block + wave; j < q_end; j += LG_WAVES)
    {
        const float qx = to_vector_register(query[j * 3 + 0]), qy = to_vector_register(query[j * 3 + 1]), qz = to_vector_register(query[j * 3 + 2]);
        u64 mine;
        const int place = nearest_in_grid<false>(grid, grid.points, grid.starts, m, k, lane, qx, qy, qz, s, mine TPK_WORK_ARG);
        if (place < k)
        {
            dist2[static_cast<int64_t>(j) * k + place] = __int_as_float(static_cast<int>(mine >> 32));
            idx[static_cast<int64_t>(j) * k + place] = static_cast<int64_t>(mine & 0xFFFFFFFFu);
        }
    }
    TPK_WORK_FLUSH
}

int launch_knn_cells(int b, int n, int m, int k, const float* query, const float* support, float* dist2, int64_t* idx, hipStream_t stream)
{
    // one workgroup per compute unit where the queries allow it (every workgroup sorts its cloud), a query per wavefront
    // at a time
    const int64_t per_cloud = std::max<int64_t>(1, std::min<int64_t>(tpk_ceil_div(n, LG_WAVES), TPK_COMPUTE_UNITS / b));
    const int per_block = static_cast<int>(tpk_ceil_div(n, per_cloud));
    const int64_t bpc = tpk_ceil_div(n, per_block);
    if (bpc * b > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    const size_t lds = lg_lds_bytes(m) + LG_WAVES * KNC_ROOM * sizeof(u64);
    const int st = tpk_allow_lds(reinterpret_cast<const void*>(&knn_cells_kernel), lds);
    if (st != TPK_OK)
        return st;
    hipLaunchKernelGGL(knn_cells_kernel, dim3(static_cast<unsigned>(bpc * b)), dim3(LG_THREADS), lds, stream, n, m, k,
                       static_cast<int>(bpc), per_block, knn_per_cell(k), query, support, dist2, idx);
    return tpk_launch_status();
}

// Larger clouds: the grid in memory, built by up to KNG_PARTS workgroups per cloud.  Two passes over the points - their box, then
// their cells' counts in LDS -, a prefix sum, and a third that writes every point's record to its cell.
constexpr int KNG_CELLS = 32768; // cells at most (their counts lie in LDS)

// Per cloud: the records [m], the cells' first places [cells + 64], the shape [LG_SHAPE], where the cloud ends [6].
struct KnnGridLayout
{
    size_t starts, shape, total;
    int cells; // at most; a multiple of 4096, the places a step of the builder's prefix sum writes
};
inline KnnGridLayout knn_grid_layout(int m, int cells)
{
    KnnGridLayout l;
    l.starts = (static_cast<size_t>(m) * sizeof(float4) + 255) & ~static_cast<size_t>(255);
    l.shape = l.starts + (static_cast<size_t>(cells) + TPK_WAVE) * sizeof(int);
    l.total = l.shape + 256;
    l.cells = cells;
    return l;
}

// Trims every axis of the grid's box, by one wavefront, to the cells outside which a 16th of the m points lies on either side
// (marginals: the points per cell along x, y, z).  The box before goes to `before`; *trimmed = whether it shrinks to KNG_KEPT or
// less, otherwise `box` stays.  With a 128th instead, clouds with 5 % of their points scattered widely stayed untrimmed: 2 x
// 100000 of those 16.0 ms, this way 1.2.  (A point sees 11 times an even cloud's points in its cell under a normal distribution, 20
// to 30 times in laser scans, hundreds in clusters: trimmed to a half from 8 times on, calls of theirs took up to twice as long.)
constexpr float KNG_CROWDED = 32.0f; // a crowded cell's points, over those that a point of an even cloud sees in its cell
constexpr float KNG_KEPT = 1.0f / 16.0f;
constexpr int KNG_ZOOMS = 8; // times at most
// Workgroups per cloud at most (a power of two).  Each goes through all its points for the box and the counts, which come out the same,
// and writes the records of its share of the cells, by stretches of KNG_STRETCH of them so that a crowd is shared too: a scattered
// record is a cache line of its own to the compute unit that writes it, a third of the builder's time.  1 x 16384 points 20.2 -> 14.5 us,
// 2 x 100000 109 -> 70 (4 parts 73, 16 parts 70).
constexpr int KNG_PARTS = 8, KNG_STRETCH = 16;

__device__ __forceinline__ void trim_box(const int* marginals, int m, const float* shape, int lane, int* box, int* before, int* trimmed)
{
    const int drop = m / 16;
    float kept = 1.0f;
    int low[3], high[3];
    for (int a = 0; a < 3; ++a)
    {
        const int cells = __float_as_int(shape[9 + a]);
        // two cells per lane
        const int n0 = marginals[a * KNG_AXIS + 2 * lane], n1 = marginals[a * KNG_AXIS + 2 * lane + 1];
        const int ahead = wave_exclusive_sum(n0 + n1), behind = m - ahead;
        const unsigned long long firsts = __ballot(ahead + n0 + n1 > drop), lasts = __ballot(behind > drop);
        const int first_lane = __builtin_ctzll(firsts), last_lane = 63 - __builtin_clzll(lasts);
        const int first = 2 * first_lane + (__builtin_amdgcn_readlane(ahead + n0, first_lane) > drop ? 0 : 1);
        const int last = 2 * last_lane + (__builtin_amdgcn_readlane(behind - n0, last_lane) > drop ? 1 : 0);
        kept *= static_cast<float>(last - first + 1) / static_cast<float>(cells);
        low[a] = first == 0 ? box[a] : lg_ordered(shape[a] + static_cast<float>(first) * shape[6 + a]);
        high[a] = last == cells - 1 ? box[3 + a] : lg_ordered(shape[a] + static_cast<float>(last + 1) * shape[6 + a]);
    }
    if (lane < 6)
    {
        before[lane] = box[lane];
        const int end = lane == 0 ? low[0] : lane == 1 ? low[1] : lane == 2 ? low[2] : lane == 3 ? high[0] : lane == 4 ? high[1] : high[2];
        if (kept <= KNG_KEPT)
            box[lane] = end;
    }
    if (lane == 0)
        *trimmed = kept <= KNG_KEPT ? 1 : 0;
}

__global__ __launch_bounds__(LG_THREADS) void knn_grid_build_kernel(int m, float per_cell, int parts, KnnGridLayout layout,
                                                                    const float* __restrict__ support, unsigned char* __restrict__ workspace)
{
    extern __shared__ __align__(16) int kng_counts[]; // [KNG_CELLS]
    __shared__ int box[6], box_before[6]; // ordered ints: min x, y, z then max x, y, z; of the zoom before
    __shared__ float shape[LG_SHAPE];
    __shared__ int wave_totals[LG_WAVES];
    __shared__ int crowded, fullest; // points in crowded cells; in the fullest of them
    __shared__ int marginals[3 * KNG_AXIS], trimmed;
    constexpr int BATCH = 8; // points in flight per lane
    const int tid = threadIdx.x;
    const int lane = tid & (TPK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / TPK_WAVE);
    const unsigned cloud = blockIdx.x / static_cast<unsigned>(parts);
    const int part = static_cast<int>(blockIdx.x - cloud * static_cast<unsigned>(parts));
    support += static_cast<int64_t>(cloud) * m * 3;
    workspace += cloud * layout.total;
    float4* __restrict__ const records = reinterpret_cast<float4*>(workspace);
    int* __restrict__ const starts = reinterpret_cast<int*>(workspace + layout.starts);

    // f(point number, x, y, z) for every point of the cloud; a lane's first BATCH points stay in its registers
    float hx[BATCH], hy[BATCH], hz[BATCH];
    auto load = [&](int first, float (&px)[BATCH], float (&py)[BATCH], float (&pz)[BATCH]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < BATCH; ++u)
        {
            const int64_t t = min(first + u * LG_THREADS, m - 1);
            px[u] = support[t * 3 + 0];
            py[u] = support[t * 3 + 1];
            pz[u] = support[t * 3 + 2];
        }
    };
    load(tid, hx, hy, hz);
    auto each = [&](auto f) __attribute__((always_inline)) {
        auto batch = [&](int first, const float (&px)[BATCH], const float (&py)[BATCH], const float (&pz)[BATCH]) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
                if (first + u * LG_THREADS < m)
                    f(first + u * LG_THREADS, px[u], py[u], pz[u]);
        };
        batch(tid, hx, hy, hz);
        for (int first = tid + BATCH * LG_THREADS; first < m; first += BATCH * LG_THREADS)
        {
            float px[BATCH], py[BATCH], pz[BATCH];
            load(first, px, py, pz);
            batch(first, px, py, pz);
        }
    };
    if (tid < 6)
        box[tid] = tid < 3 ? 0x7FFFFFFF : INT_MIN;
    const float inf = __builtin_inff();
    float lows[3] = {inf, inf, inf}, highs[3] = {-inf, -inf, -inf};
    each([&](int, float x, float y, float z) {
        const float v[3] = {x, y, z};
#pragma unroll
        for (int a = 0; a < 3; ++a)
        {
            const bool finite = fabsf(v[a]) < inf;
            lows[a] = lg_min(lows[a], finite ? v[a] : inf);
            highs[a] = lg_max(highs[a], finite ? v[a] : -inf);
        }
    });
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 3; ++a)
    {
        const int low = ~wave_max_i32(~lg_ordered(lows[a])), high = wave_max_i32(lg_ordered(highs[a]));
        if (lane == 0)
        {
            atomicMin(&box[a], low);
            atomicMax(&box[3 + a], high);
        }
    }
    __syncthreads();
    float ends[6]; // the cloud's: min x, y, z then max x, y, z
#pragma unroll
    for (int a = 0; a < 6; ++a)
        ends[a] = lg_unordered(box[a]);

    float lo[3], inv[3];
    int cx, cy, cz;
    auto cell_of = [&](float x, float y, float z) __attribute__((always_inline)) {
        return lg_cell((x - lo[0]) * inv[0], cx) + cx * (lg_cell((y - lo[1]) * inv[1], cy) + cy * lg_cell((z - lo[2]) * inv[2], cz));
    };
    // Uneven clouds.  A few points far out leave all others in a cell or two, whose queries would walk the whole cloud.  Where half of
    // the points lie in such cells, and most of the box holds hardly a point, the grid is laid over the rest of the box and its
    // outermost cells take what lies beyond.  8 x 16384 points, one of them at 1000 cloud sizes, k = 16: 2040 us, this way 232.
    const int crowd = static_cast<int>(KNG_CROWDED * (per_cell + 1.0f));
    int fullest_before = m;
    for (int zooms = 0;; ++zooms)
    {
        if (wave == 0)
            lg_shape(box, m, per_cell, KNG_AXIS, layout.cells, lane, shape);
        __syncthreads();
#pragma unroll
        for (int a = 0; a < 3; ++a)
        {
            lo[a] = shape[a];
            inv[a] = shape[3 + a];
        }
        cx = __float_as_int(shape[9]), cy = __float_as_int(shape[10]), cz = __float_as_int(shape[11]);
        const int steps = (cx * cy * cz + 4 * LG_THREADS - 1) / (4 * LG_THREADS); // of the prefix sum, four cells per lane
        for (int c = tid; c < steps * LG_THREADS; c += LG_THREADS)
            reinterpret_cast<int4*>(kng_counts)[c] = make_int4(0, 0, 0, 0);
        if (tid == 0)
            crowded = fullest = 0;
        __syncthreads();
        each([&](int, float x, float y, float z) { atomicAdd(&kng_counts[cell_of(x, y, z)], 1); });
        __syncthreads();
        int placed = 0; // points in the cells of the steps before
        for (int step = 0; step < steps; ++step)
        {
            int4* const four = reinterpret_cast<int4*>(kng_counts) + step * LG_THREADS + tid;
            const int4 c4 = *four;
            const int own = c4.x + c4.y + c4.z + c4.w;
            const int in_crowds = (c4.x > crowd ? c4.x : 0) + (c4.y > crowd ? c4.y : 0) + (c4.z > crowd ? c4.z : 0) + (c4.w > crowd ? c4.w : 0);
            const int before = wave_exclusive_sum(own);
            if (lane == TPK_WAVE - 1)
                wave_totals[wave] = before + own;
            __syncthreads();
            const int total = lane < LG_WAVES ? wave_totals[lane] : 0;
            const int totals_before = wave_exclusive_sum(total);
            int at = placed + __builtin_amdgcn_readlane(totals_before, wave) + before;
            placed += __builtin_amdgcn_readlane(totals_before + total, LG_WAVES - 1);
            int4 s4;
            s4.x = at;
            s4.y = at += c4.x;
            s4.z = at += c4.y;
            s4.w = at += c4.z;
            *four = s4;
            if (part == 0)
                reinterpret_cast<int4*>(starts)[step * LG_THREADS + tid] = s4; // (also those behind the last cell: the end)
            if (in_crowds != 0)
            {
                atomicAdd(&crowded, in_crowds);
                atomicMax(&fullest, max(max(c4.x, c4.y), max(c4.z, c4.w)));
            }
            __syncthreads();
        }
        if (tid == 0 && part == 0)
            starts[steps * 4 * LG_THREADS] = m;
        // (from here on everything is the same for the whole workgroup)
        const int fullest_now = fullest;
        if (zooms > KNG_ZOOMS || crowded <= m / 2)
            break;
        if (zooms == KNG_ZOOMS || fullest_now > fullest_before)
        {
            if (fullest_now <= fullest_before)
                break;
            // the last zoom made it worse: back to the box before
            if (tid < 6)
                box[tid] = box_before[tid];
            zooms = KNG_ZOOMS;
            __syncthreads();
            continue;
        }
        fullest_before = fullest_now;
        for (int c = tid; c < 3 * KNG_AXIS; c += LG_THREADS)
            marginals[c] = 0;
        __syncthreads();
        // (the counts of planes and rows are differences of the prefix sums; neighbouring lanes add to neighbouring places)
        const int cells = cx * cy * cz;
        auto count_of = [&](int first, int end) __attribute__((always_inline)) { return (end < cells ? kng_counts[end] : m) - kng_counts[first]; };
        const float per_row = __builtin_amdgcn_rcpf(static_cast<float>(cx)), per_plane = __builtin_amdgcn_rcpf(static_cast<float>(cy));
        for (int c = tid; c < cells; c += LG_THREADS)
        {
            const int count = count_of(c, c + 1);
            if (count != 0)
                atomicAdd(&marginals[c - cx * static_cast<int>((static_cast<float>(c) + 0.5f) * per_row)], count);
        }
        for (int row = tid; row < cy * cz; row += LG_THREADS)
            atomicAdd(&marginals[KNG_AXIS + row - cy * static_cast<int>((static_cast<float>(row) + 0.5f) * per_plane)], count_of(row * cx, row * cx + cx));
        if (tid < cz)
            marginals[2 * KNG_AXIS + tid] = count_of(tid * cx * cy, (tid + 1) * cx * cy);
        __syncthreads();
        if (wave == 0)
            trim_box(marginals, m, shape, lane, box, box_before, &trimmed);
        __syncthreads();
        if (!trimmed)
            break;
    }
    if (tid < LG_SHAPE && part == 0)
        reinterpret_cast<float*>(workspace + layout.shape)[tid] = shape[tid];
    if (tid < 3 && part == 0)
    {
        // where the cloud ends, in cells
        const float low = tid == 0 ? ends[0] : tid == 1 ? ends[1] : ends[2], high = tid == 0 ? ends[3] : tid == 1 ? ends[4] : ends[5];
        float* const behind = reinterpret_cast<float*>(workspace + layout.shape) + LG_SHAPE;
        behind[tid] = fminf((low - shape[tid]) * shape[3 + tid], 0.0f);
        behind[3 + tid] = fmaxf((high - shape[tid]) * shape[3 + tid], static_cast<float>(__float_as_int(shape[9 + tid])));
    }
    each([&](int t, float x, float y, float z) {
        const int c = cell_of(x, y, z);
        if (((c / KNG_STRETCH) & (parts - 1)) == part)
            records[atomicAdd(&kng_counts[c], 1)] = make_float4(x, y, z, __int_as_float(t));
    });
}

// The shape of a grid in memory, as its builder left it.
__device__ __forceinline__ void knn_grid_read(LdsGrid& grid, const float* __restrict__ shape)
{
#pragma unroll
    for (int a = 0; a < 3; ++a)
    {
        grid.lo[a] = shape[a];
        grid.inv[a] = shape[3 + a];
        grid.width[a] = shape[6 + a];
        grid.cells[a] = __float_as_int(shape[9 + a]);
        grid.below[a] = shape[LG_SHAPE + a];
        grid.above[a] = shape[LG_SHAPE + 3 + a];
    }
    grid.volume = shape[12];
}

__global__ __launch_bounds__(KNN_THREADS) void knn_grid_search_kernel(int64_t queries, int n, int m, int k, KnnGridLayout layout,
                                                                      const float* __restrict__ query, const unsigned char* __restrict__ workspace,
                                                                      float* __restrict__ dist2, int64_t* __restrict__ idx)
{
    __shared__ u64 keys[KNN_THREADS / TPK_WAVE][KNC_ROOM];
    const int lane = threadIdx.x & (TPK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TPK_WAVE);
    const int64_t j = static_cast<int64_t>(xcd_local_block(blockIdx.x, gridDim.x)) * (KNN_THREADS / TPK_WAVE) + wave;
    if (j >= queries)
        return; // (no workgroup barrier anywhere in this kernel)
    workspace += (j / n) * layout.total;
    const float qx = to_vector_register(query[j * 3 + 0]), qy = to_vector_register(query[j * 3 + 1]), qz = to_vector_register(query[j * 3 + 2]);
    TPK_WORK_DECL
    LdsGrid grid;
    knn_grid_read(grid, reinterpret_cast<const float*>(workspace + layout.shape));
    Survivors s;
    s.keys = keys[wave];
    s.lane = lane;
    s.k = k;
    u64 mine;
    const int place = nearest_in_grid<true>(grid, reinterpret_cast<const float4*>(workspace), reinterpret_cast<const int*>(workspace + layout.starts), m, k,
                                      lane, qx, qy, qz, s, mine TPK_WORK_ARG);
    if (place < k)
    {
        dist2[j * k + place] = __int_as_float(static_cast<int>(mine >> 32));
        idx[j * k + place] = static_cast<int64_t>(mine & 0xFFFFFFFFu);
    }
    TPK_WORK_FLUSH
}

// Four queries of a cloud per wavefront, 16 lanes each, up to 16 neighbours.  A query looks at a block of cells - its own if that holds 2k
// points, the eight whose common corner is nearest to it if they hold 4k, else the 27 around it -, has the block's first 16 * PER
// points in its lanes' registers, PER each, and looks for a distance with k to k + KNQ_SPARE of them within it, all four at once.  The
// rest of the block, and then the cells outside that the ball around the k nearest so far touches, are walked for points within
// reach, 16 a step; longer walks by the whole wavefront, 64 a step, one query after the other.  Queries that need a larger block, with
// too many equal distances or more than KNQ_PIECES rows of cells outside are left to nearest_in_grid.
// Bound by instruction issue (8 x 16384 even, k = 16: 1010 vector instructions per wavefront, 252 per query, 55 of the kernel's 59 us), most of
// which nearest_in_grid spends whatever the number of candidates: a wavefront that serves one query has 86 of them in an even cloud (k = 16),
// a third of whose queries look outside.  Calls of k = 4 / 16, as many queries as points, a wavefront a query and this way, us:
//                                            8 x 4099                8 x 16384                2 x 100000                 1 x 33000
//     even                                30 / 35 -> 24 / 29       87 / 106 -> 58 / 70     219 / 240 -> 136 / 150      61 / 65 -> 44 / 46
//     sphere                              33 / 35 -> 25 / 30      104 / 118 -> 64 / 75     254 / 298 -> 160 / 194      66 / 71 -> 47 / 49
//     clusters of sigma 0.05              39 / 53 -> 32 / 50      125 / 192 -> 85 / 156    320 / 413 -> 246 / 325      75 / 97 -> 57 / 85
//     clusters of sigma 0.02              44 / 56 -> 41 / 59      171 / 270 -> 147 / 253   566 / 713 -> 454 / 633      98 / 133 -> 89 / 131
//     clusters of sigma 0.003             51 / 57 -> 55 / 63      338 / 365 -> 278 / 344  2234 / 2360 -> 1654 / 1787  194 / 199 -> 179 / 199
//     laser scan (radius 1.5 to 50)       35 / 44 -> 31 / 47      102 / 138 -> 78 / 120    279 / 319 -> 206 / 256      67 / 79 -> 53 / 65
//     queries 300 cloud sizes away        38 / 43 -> 45 / 37      117 / 135 -> 72 / 107    250 / 287 -> 145 / 187      68 / 67 -> 48 / 49
//     the same along one axis             99 / 105 -> 111 / 100   692 / 619 -> 708 / 563  1946 / 2201 -> 1914 / 2300  307 / 260 -> 376 / 291
//     queries over 3 times the width      39 / 45 -> 48 / 48      128 / 155 -> 124 / 157   272 / 346 -> 208 / 352      76 / 83 -> 77 / 85
// What is still slower are small calls whose queries have long walks, which a quarter of the wavefronts then take one after the other.
// (Without the eight cells: 8 x 16384 on a sphere, k = 16, 111; without the walks by the wavefront in clusters 273; with four wavefronts
// per SIMD instead of six, which spill two registers, 77 to 81 even; seven and eight spill 14 and 33 and take 82 and more.)  k = 32, with 16
// points a lane, was 8 to 13 % faster in even clouds and 10 to 20 % slower in clusters.
// Built, measured, dropped: queries that are given up, or have hundreds of points to walk through or are far away, handed to a launch of
// their own with a wavefront a query (8 x 4099, k = 16, even 30, clusters of sigma 0.003 80 to 105, far 53); queries that are given up
// shared among a workgroup's wavefronts, behind a barrier (8 x 16384, k = 4 / 16, even 67 / 79, queries over 3 times the width 136 / 169).
constexpr int KNQ_MAX_K = 16;
// Queries from which on: with fewer the four wait for each other while wavefronts' places are empty - at six per SIMD there are 6144, 24576
// queries -, and what uneven clouds and queries outside lose outweighs what even ones gain.  k = 4 / 16, time over a wavefront a query's, even,
// clusters of sigma 0.05 and 0.003, queries over 3 times the width: 1 x 9000 0.98 / 1.00, 1.01 / 1.10, 1.17 / 1.28, 1.31 / 1.51; 4 x 5000 0.90 / 0.88,
// 0.93 / 0.98, 1.09 / 1.13, 1.23 / 1.20; 7 x 4099 0.89 / 0.86, 0.90 / 0.99, 1.13 / 1.16, 1.19 / 1.09; 2 x 16000 0.88 / 0.87, 0.87 / 0.97, 0.99 / 1.09,
// 1.20 / 1.25; 8 x 4099 0.79 / 0.81, 0.81 / 0.93, 1.08 / 1.11, 1.20 / 1.06; 8 x 16384 0.66 / 0.66, 0.68 / 0.81, 0.83 / 0.94, 0.96 / 1.01.
constexpr int64_t KNQ_LEAST = 32768;
constexpr int KNQ_GROUP = 16, KNQ_QUERIES = TPK_WAVE / KNQ_GROUP;
constexpr int KNQ_OWN = 2, KNQ_EIGHT = 4; // (3 for the eight: within 2 %)
constexpr int KNQ_SPARE = 16;  // (8: 1 to 3 % faster, but then nothing separates the 8 nearest on a lattice, where 7 and 19 points lie within a distance)
constexpr int KNQ_TRIES = 12;  // guesses of the distance
constexpr int KNQ_FULL = 48;   // keys kept between two steps at most; a step adds up to 64
constexpr int KNQ_LONG = 64;   // points of a walk by 16 lanes at most (112: 2 % slower in clusters)
// The guess after which the distance of a selection is looked for between the nearest and the farthest candidate: seen from far away all
// are about equally distant, which no estimate by volume finds.  (8 x 16384, queries 300 cloud sizes away, k = 16: 189 -> 107 us, a
// quarter of them were given up after 12 guesses; a wavefront a query 135.  One guess earlier: 106, and 3 % slower on laser scans.)
constexpr int KNQ_SPREAD = 2;
// A single query with more rows of cells than this is given up, since the whole wavefront goes through them four times as fast; not where
// most of the four have as many (8 x 16384, queries 300 cloud sizes away along one axis, k = 4 / 16: 833 / 761 -> 710 / 560 us).
constexpr int KNQ_PIECES = 256, KNQ_TOGETHER = 3;

// Puts the first cnt (<= 16 * HELD) keys of every query of the wavefront in ascending order, of which the k first stay.
template <int HELD>
__device__ __forceinline__ void order_kept(u64* mine, int cnt, int k, int sub)
{
    u64 key[HELD];
    int rank[HELD];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (sub < 4)
        mine[cnt + sub] = ~0ull; // (read four at a time)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int h = 0; h < HELD; ++h)
    {
        key[h] = h * KNQ_GROUP + sub < cnt ? mine[h * KNQ_GROUP + sub] : ~0ull;
        rank[h] = 0;
    }
    for (int i = 0; i < cnt; i += 4)
    {
#pragma unroll
        for (int u = 0; u < 4; ++u)
        {
            const u64 other = mine[i + u];
#pragma unroll
            for (int h = 0; h < HELD; ++h)
                rank[h] += other < key[h] ? 1 : 0;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int h = 0; h < HELD; ++h)
        if (h * KNQ_GROUP + sub < cnt && rank[h] < k)
            mine[rank[h]] = key[h];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// The same for one query's keys by the whole wavefront, up to two a lane.
__device__ __forceinline__ void order_kept_by_wave(u64* mine, int cnt, int k, int lane)
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane < 4)
        mine[cnt + lane] = ~0ull;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const u64 key0 = lane < cnt ? mine[lane] : ~0ull, key1 = TPK_WAVE + lane < cnt ? mine[TPK_WAVE + lane] : ~0ull;
    int rank0 = 0, rank1 = 0;
    for (int i = 0; i < cnt; i += 4)
    {
#pragma unroll
        for (int u = 0; u < 4; ++u)
        {
            const u64 other = mine[i + u];
            rank0 += other < key0 ? 1 : 0;
            rank1 += other < key1 ? 1 : 0;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane < cnt && rank0 < k)
        mine[rank0] = key0;
    if (TPK_WAVE + lane < cnt && rank1 < k)
        mine[rank1] = key1;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// The smallest, or (LARGEST) the largest of the row's 16 values >= 0.
template <bool LARGEST>
__device__ __forceinline__ float row_extreme(float v)
{
    // (floats >= 0 order like their bits)
    int s = __float_as_int(v);
    auto with = [&](int turned) __attribute__((always_inline)) { s = LARGEST ? max(s, turned) : min(s, turned); };
    with(__builtin_amdgcn_update_dpp(0, s, 0x128, 0xF, 0xF, true)); // row_ror:8
    with(__builtin_amdgcn_update_dpp(0, s, 0x124, 0xF, 0xF, true));
    with(__builtin_amdgcn_update_dpp(0, s, 0x122, 0xF, 0xF, true));
    with(__builtin_amdgcn_update_dpp(0, s, 0x121, 0xF, 0xF, true));
    return __int_as_float(s);
}

template <int PER>
__global__ __launch_bounds__(KNN_THREADS, 6) void knn_grid_four_kernel(int n, int m, int k, unsigned blocks_per_cloud, KnnGridLayout layout,
                                                                    const float* __restrict__ query, const unsigned char* __restrict__ workspace,
                                                                    float* __restrict__ dist2, int64_t* __restrict__ idx)
{
    constexpr int WAVES = KNN_THREADS / TPK_WAVE;
    constexpr int MOST = PER * KNQ_GROUP;                              // a query's candidates
    constexpr int ROOM = KNQ_FULL + TPK_WAVE + 4;
    static_assert(MOST <= 256 && KNQ_MAX_K + KNQ_SPARE <= KNQ_FULL, "a byte holds a place, the selected keys fit");
    __shared__ u64 keys[WAVES][KNC_ROOM];
    __shared__ u64 kept[WAVES][KNQ_QUERIES][ROOM];
    __shared__ unsigned marks[WAVES][KNQ_QUERIES][MOST / 4];
    const int lane = threadIdx.x & (TPK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TPK_WAVE);
    const unsigned block = xcd_local_block(blockIdx.x, gridDim.x);
    const unsigned cloud = block / blocks_per_cloud;
    const int64_t j0 = (static_cast<int64_t>(block - cloud * blocks_per_cloud) * WAVES + wave) * KNQ_QUERIES;
    if (j0 >= n)
        return; // (no workgroup barrier anywhere in this kernel)
    workspace += cloud * layout.total;
    const float* __restrict__ const shape = reinterpret_cast<const float*>(workspace + layout.shape);
    const int q0 = static_cast<int>(j0);
    const int group = lane / KNQ_GROUP, sub = lane % KNQ_GROUP;
    const bool real = q0 + group < n;
    query += static_cast<int64_t>(cloud) * n * 3;
    dist2 += static_cast<int64_t>(cloud) * n * k;
    idx += static_cast<int64_t>(cloud) * n * k;
    const int64_t j = real ? q0 + group : q0;
    const float q[3] = {query[j * 3 + 0], query[j * 3 + 1], query[j * 3 + 2]};
    const float4* __restrict__ const points = reinterpret_cast<const float4*>(workspace);
    const int* __restrict__ const starts = reinterpret_cast<const int*>(workspace + layout.starts);
    TPK_WORK_DECL
    LdsGrid grid;
    knn_grid_read(grid, shape);
    Survivors s;
    s.keys = keys[wave];
    s.lane = lane;
    s.k = k;

    // ---- the block's rows of cells, one per lane ----
    const int cx = grid.cells[0], cy = grid.cells[1];
    float t[3]; // in cells
    int c[3], low[3], high[3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
    {
        t[a] = (q[a] - grid.lo[a]) * grid.inv[a];
        c[a] = lg_cell(t[a], grid.cells[a]);
    }
    // The rows of the 27 cells around the query and of the eight whose common corner is nearest to it: both looked up at once.
    auto rows_of = [&](const int* from, const int* to, int& start, int& size) __attribute__((always_inline)) {
        const int ny = to[1] - from[1] + 1, rows = ny * (to[2] - from[2] + 1); // up to 9
        start = size = 0;
        if (sub < rows)
        {
            int row = sub + (c[1] - from[1]) + ny * (c[2] - from[2]); // (the query's own row first)
            row -= row >= rows ? rows : 0;
            const int iz = (row >= ny ? 1 : 0) + (row >= 2 * ny ? 1 : 0);
            const int c0 = from[0] + cx * ((from[1] + row - iz * ny) + cy * (from[2] + iz));
            start = starts[c0];
            size = starts[c0 + to[0] - from[0] + 1] - start;
        }
    };
    int low8[3], high8[3], start, size, start8, size8;
#pragma unroll
    for (int a = 0; a < 3; ++a)
    {
        low[a] = max(c[a] - 1, 0), high[a] = min(c[a] + 1, grid.cells[a] - 1);
        const bool upper = t[a] - static_cast<float>(c[a]) >= 0.5f;
        low8[a] = upper ? c[a] : low[a], high8[a] = upper ? high[a] : c[a];
    }
    rows_of(low, high, start, size);
    rows_of(low8, high8, start8, size8);
    const int own = c[0] + cx * (c[1] + cy * c[2]);
    const int own_start = starts[own], own_size = starts[own + 1] - own_start;
    const bool one = own_size >= KNQ_OWN * k, eight = row_last(row_exclusive_sum(size8) + size8, lane) >= KNQ_EIGHT * k;
    start = one ? own_start : eight ? start8 : start;
    size = one ? (sub == 0 ? own_size : 0) : eight ? size8 : size;
#pragma unroll
    for (int a = 0; a < 3; ++a)
    {
        low[a] = one ? c[a] : eight ? low8[a] : low[a];
        high[a] = one ? c[a] : eight ? high8[a] : high[a];
    }
    const int cells = (high[0] - low[0] + 1) * (high[1] - low[1] + 1) * (high[2] - low[2] + 1);
    const int before = row_exclusive_sum(size);
    const int total = row_last(before + size, lane);
    bool good = real && total >= k, done = false;
    if (__ballot(good) != 0)
    {
        // ---- its points: every row's lane marks the place of its first one, a running maximum finds the others' row ----
        const int origin = start - before; // candidate i of a row's lane lies at origin + i
        unsigned* const my_marks = marks[wave][group];
        unsigned char* const mark = reinterpret_cast<unsigned char*>(my_marks);
#pragma unroll
        for (int i = 0; i < PER / 4; ++i)
            my_marks[i * KNQ_GROUP + sub] = 0;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (good && size > 0 && before < MOST)
            mark[before] = static_cast<unsigned char>(sub);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        float4 p[PER];
        int carried = 0;
#pragma unroll
        for (int i = 0; i < PER; ++i)
        {
            const int at = i * KNQ_GROUP + sub;
            const int row = max(row_inclusive_max(mark[at]), carried);
            carried = row_last(row, lane);
            const int place = __builtin_amdgcn_ds_bpermute((group * KNQ_GROUP + row) * 4, origin) + at;
            p[i] = points[good && at < total ? place : 0];
        }
        float d[PER];
#pragma unroll
        for (int i = 0; i < PER; ++i)
        {
            TPK_WORK_ADD(1);
            d[i] = good && i * KNQ_GROUP + sub < total ? tpk_dist2(q[0], q[1], q[2], p[i].x, p[i].y, p[i].z) : __builtin_inff();
        }

        // ---- a distance with k .. k + KNQ_SPARE of them within it (as Survivors::select) ----
        const float target = static_cast<float>(k + KNQ_SPARE / 2);
        float guess = s.volume_ratio(0.2387f * grid.volume * static_cast<float>(cells) * __builtin_amdgcn_rcpf(static_cast<float>(total)) * target);
        Bracket bracket;
        int within = 0, count = 0, held = 0;
        for (int tries = 0;; ++tries)
        {
            count = 0;
#pragma unroll
            for (int i = 0; i < PER; ++i)
                count += d[i] <= guess && d[i] < __builtin_inff() ? 1 : 0;
            within = row_exclusive_sum(count);
            held = row_last(within + count, lane);
            const bool fits = held >= k && held <= k + KNQ_SPARE;
            if (tries == KNQ_TRIES || __ballot(good && !fits) == 0)
            {
                good = good && fits;
                break;
            }
            const float estimate = guess * s.volume_ratio(target * __builtin_amdgcn_rcpf(fmaxf(static_cast<float>(held), 0.5f)));
            float next = bracket.next(guess, held < k, estimate, tries);
            if (tries == KNQ_SPREAD)
            {
                float nearest = __builtin_inff(), farthest = 0.0f;
#pragma unroll
                for (int i = 0; i < PER; ++i)
                {
                    nearest = fminf(nearest, d[i]);
                    farthest = d[i] < __builtin_inff() ? fmaxf(farthest, d[i]) : farthest;
                }
                nearest = row_extreme<false>(nearest);
                farthest = row_extreme<true>(farthest);
                const int candidates = min(total, MOST);
                const float between = nearest + (farthest - nearest) * (target * __builtin_amdgcn_rcpf(static_cast<float>(candidates)));
                const bool all = candidates <= k + KNQ_SPARE; // (these fit)
                next = all ? farthest : between > bracket.lo && between < bracket.hi ? between : next;
                bracket.lo = fmaxf(bracket.lo, nearest * 0.9999999f); // (the float below `nearest`: none lies within it)
                bracket.hi = all ? bracket.hi : fminf(bracket.hi, farthest);
            }
            guess = fits ? guess : next;
        }

        u64* const mine = kept[wave][group];
        int cnt = good ? held : 0; // kept so far
        float reach = guess;       // the k-th lies within it
        if (good)
        {
            int at = within;
#pragma unroll
            for (int i = 0; i < PER; ++i)
                if (d[i] <= guess && d[i] < __builtin_inff())
                    mine[at++] = knn_key(d[i], __float_as_int(p[i].w));
        }
        auto order = [&]() __attribute__((always_inline)) {
            if (rows_max(cnt) <= 2 * KNQ_GROUP)
                order_kept<2>(mine, cnt, k, sub);
            else
                order_kept<(KNQ_FULL + KNQ_GROUP) / KNQ_GROUP>(mine, cnt, k, sub);
            if (cnt >= k)
            {
                cnt = k;
                reach = __int_as_float(static_cast<int>(mine[k - 1] >> 32));
            }
        };
        // The candidates from c0 on of the rows of cells that a query's lanes hold (single: its first lane alone).
        auto walk = [&](int start, int size, int before, int total, int c0, bool single) __attribute__((always_inline)) {
            const int origin = start - before;
            unsigned long long longer = __ballot(total - c0 > KNQ_LONG && sub == 0);
            while (longer != 0)
            {
                const int first = __builtin_ctzll(longer); // the query's first lane
                longer &= longer - 1;
                unsigned char* const mark64 = reinterpret_cast<unsigned char*>(marks[wave][0]);
                u64* const its = kept[wave][first / KNQ_GROUP];
                const int its_total = tpk_read_lane(total, first);
                const float x = to_vector_register(tpk_read_lane(q[0], first)), y = to_vector_register(tpk_read_lane(q[1], first)),
                            z = to_vector_register(tpk_read_lane(q[2], first));
                const bool row_here = first / KNQ_GROUP == group && size > 0;
                int its_cnt = tpk_read_lane(cnt, first);
                float its_reach = tpk_read_lane(reach, first);
                // (no looking up whose a candidate is where there is one row: clusters of sigma 0.003, 8 x 16384, 423 -> 342 us)
                const bool its_single = tpk_read_lane(single ? 1 : 0, first) != 0;
                const int its_origin = tpk_read_lane(origin, first);
                auto fetch = [&](int c) __attribute__((always_inline)) {
                    if (its_single)
                        return points[c + lane < its_total ? its_origin + c + lane : 0];
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    mark64[lane] = 0;
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    if (row_here && before < c + TPK_WAVE && before + size > c)
                        mark64[max(before - c, 0)] = static_cast<unsigned char>(sub);
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    const int place = __builtin_amdgcn_ds_bpermute((first + wave_inclusive_max_i32(mark64[lane])) * 4, origin) + c + lane;
                    return points[c + lane < its_total ? place : 0];
                };
                float4 ahead = fetch(c0);
                for (int c = c0; c < its_total; c += TPK_WAVE)
                {
                    const float4 p = ahead;
                    if (c + TPK_WAVE < its_total)
                        ahead = fetch(c + TPK_WAVE);
                    TPK_WORK_ADD(1);
                    const float d = tpk_dist2(x, y, z, p.x, p.y, p.z);
                    const bool hit = c + lane < its_total && d <= its_reach && d < __builtin_inff();
                    const unsigned long long all = __ballot(hit);
                    if (all == 0)
                        continue;
                    if (hit)
                        its[its_cnt + static_cast<int>(tpk_prefix_count(all))] = knn_key(d, __float_as_int(p.w));
                    its_cnt += __builtin_popcountll(all);
                    if (its_cnt > KNQ_FULL)
                    {
                        order_kept_by_wave(its, its_cnt, k, lane);
                        its_cnt = k;
                        its_reach = tpk_read_lane(__int_as_float(static_cast<int>(its[k - 1] >> 32)), 0);
                    }
                }
                cnt = first / KNQ_GROUP == group ? its_cnt : cnt;
                reach = first / KNQ_GROUP == group ? its_reach : reach;
            }
            total = total - c0 > KNQ_LONG ? 0 : total;
            const int most = rows_max(total);
            auto fetch = [&](int c0) __attribute__((always_inline)) {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                mark[sub] = 0;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                if (size > 0 && before < c0 + KNQ_GROUP && before + size > c0)
                    mark[max(before - c0, 0)] = static_cast<unsigned char>(sub);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                const int place = __builtin_amdgcn_ds_bpermute((group * KNQ_GROUP + row_inclusive_max(mark[sub])) * 4, origin) + c0 + sub;
                return points[c0 + sub < total ? place : 0];
            };
            if (c0 >= most)
                return;
            float4 ahead = fetch(c0);
            for (; c0 < most; c0 += KNQ_GROUP)
            {
                const float4 p = ahead;
                if (c0 + KNQ_GROUP < most)
                    ahead = fetch(c0 + KNQ_GROUP);
                TPK_WORK_ADD(1);
                const float d = tpk_dist2(q[0], q[1], q[2], p.x, p.y, p.z);
                const bool hit = c0 + sub < total && d <= reach && d < __builtin_inff();
                const unsigned long long all = __ballot(hit);
                if (all == 0)
                    continue;
                const unsigned here = static_cast<unsigned>(all >> (group * KNQ_GROUP)) & 0xffffu;
                if (hit)
                    mine[cnt + __builtin_popcount(here & ((1u << sub) - 1u))] = knn_key(d, __float_as_int(p.w));
                cnt += __builtin_popcount(here);
                if (__ballot(cnt > KNQ_FULL) != 0)
                    order();
            }
        };
        walk(start, size, before, good ? total : 0, MOST, one);
        order();

        // ---- the cells outside the block that the ball around the k-th touches (the ends as in nearest_in_grid) ----
        const float bound = reach;
        const float radius = __builtin_amdgcn_sqrtf(bound) * 1.00001f;
        int from[3], to[3];
        bool inside = true;
#pragma unroll
        for (int a = 0; a < 3; ++a)
        {
            const float span = radius * grid.inv[a] + 1e-5f * (fabsf(t[a]) + static_cast<float>(KNG_AXIS));
            from[a] = lg_cell(t[a] - span, grid.cells[a]);
            to[a] = lg_cell(t[a] + span, grid.cells[a]);
            inside = inside && from[a] >= low[a] && to[a] <= high[a];
        }
        if (!inside)
            ball_rows_of_far_query(grid, t, bound, from, to);
        const int wide = to[1] - from[1] + 1, pieces = 2 * wide * (to[2] - from[2] + 1); // (two for a row that crosses the block)
        const int long_lists = __builtin_popcountll(__ballot(good && !inside && pieces > KNQ_PIECES && sub == 0));
        done = good && (inside || pieces <= KNQ_PIECES || long_lists >= KNQ_TOGETHER);
        const bool wider = done && !inside;
        for (int piece0 = 0; __ballot(wider && piece0 < pieces) != 0; piece0 += KNQ_GROUP)
        {
            const int e = piece0 + sub;
            int start = 0, size = 0;
            if (wider && e < pieces)
            {
                const bool right = e & 1;
                const int row = e >> 1;
                const int iz = static_cast<int>((static_cast<float>(row) + 0.5f) * __builtin_amdgcn_rcpf(static_cast<float>(wide)));
                const int y = from[1] + row - iz * wide, z = from[2] + iz;
                const bool crosses = y >= low[1] && y <= high[1] && z >= low[2] && z <= high[2];
                int x_from, x_to;
                const bool touched = ball_row<true>(grid, t, bound, y, z, x_from, x_to);
                const int x0 = right ? max(high[0] + 1, x_from) : x_from;
                const int x1 = right ? (crosses ? x_to : -1) : (crosses ? min(low[0] - 1, x_to) : x_to);
                if (touched && x1 >= x0)
                {
                    const int c0 = cx * (y + cy * z);
                    start = starts[c0 + x0];
                    size = starts[c0 + x1 + 1] - start;
                }
            }
            const int before = row_exclusive_sum(size);
            walk(start, size, before, row_last(before + size, lane), 0, false);
        }
        if (__ballot(cnt > k) != 0)
            order();
    }

    if (done)
        for (int e = sub; e < k; e += KNQ_GROUP)
        {
            const u64 key = kept[wave][group][e];
            dist2[j * k + e] = __int_as_float(static_cast<int>(key >> 32));
            idx[j * k + e] = static_cast<int64_t>(key & 0xFFFFFFFFu);
        }

    unsigned long long left = __ballot(real && !done && sub == 0);
    while (left != 0)
    {
        const int from = __builtin_ctzll(left);
        left &= left - 1;
        u64 mine;
        const int place = nearest_in_grid<true>(grid, points, starts, m, k, lane, to_vector_register(tpk_read_lane(q[0], from)),
                                                to_vector_register(tpk_read_lane(q[1], from)), to_vector_register(tpk_read_lane(q[2], from)),
                                                s, mine TPK_WORK_ARG);
        const int64_t out = static_cast<int64_t>(q0 + from / KNQ_GROUP) * k;
        if (place < k)
        {
            dist2[out + place] = __int_as_float(static_cast<int>(mine >> 32));
            idx[out + place] = static_cast<int64_t>(mine & 0xFFFFFFFFu);
        }
    }
    TPK_WORK_FLUSH
}

// The grid in LDS saves a launch and the few workgroups per cloud in front of the search; the grid in memory leaves room for
// twice as many wavefronts.  (16 queries per wavefront of the chip: k = 16, 4 x 4000: 25.3 and 26.3 us, 8 x 4099: 42.8 and
// 39.6 us, 8 x 8192: 73.8 and 65.4 us.)
constexpr int64_t KNC_LDS_QUERIES = 16384;
inline bool knn_in_lds(int b, int m, int n, bool workspace)
{
    return m <= LG_MAX_POINTS && (static_cast<int64_t>(b) * n <= KNC_LDS_QUERIES || !workspace);
}

size_t knn_grid_workspace_bytes(int b, int m, int n)
{
    return b > 0 && n > 0 && !knn_in_lds(b, m, n, true) ? b * knn_grid_layout(m, KNG_CELLS).total : 0;
}

// The cells of the grid that a workspace has room for (0: none).  One for the search over curve-ordered cells
// (tpk_knn_workspace_bytes) holds 18.5 bytes per point, which leaves a smaller cloud fewer than KNG_CELLS beside its records, but
// hardly fewer than it has use for: 1000 queries in a cloud of 12000 points, k = 4 and 16: lists over curve-ordered cells 224 and
// 671 us (lists of 32 entries 1505), this way 24.
int knn_grid_cells(int b, int m, int n, size_t workspace_bytes)
{
    if (workspace_bytes >= knn_grid_workspace_bytes(b, m, n))
        return KNG_CELLS;
    const size_t lists = tpk_grid_knn_workspace_bytes(b, n, m);
    if (lists == 0 || workspace_bytes < lists)
        return 0;
    int cells = KNG_CELLS;
    while (cells > 0 && b * knn_grid_layout(m, cells).total > workspace_bytes)
        cells -= 4 * LG_THREADS;
    return cells;
}

int launch_knn_grid(int b, int n, int m, int k, int cells, const float* query, const float* support, float* dist2, int64_t* idx, void* workspace,
                    hipStream_t stream)
{
    const int64_t queries = static_cast<int64_t>(b) * n, blocks = tpk_ceil_div(queries, KNN_THREADS / TPK_WAVE);
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    if (reinterpret_cast<uintptr_t>(workspace) & 255u)
        return TPK_ERR_WORKSPACE;
    const size_t lds = KNG_CELLS * sizeof(int);
    const int st = tpk_allow_lds(reinterpret_cast<const void*>(&knn_grid_build_kernel), lds);
    if (st != TPK_OK)
        return st;
    const KnnGridLayout layout = knn_grid_layout(m, cells);
    unsigned char* const w = static_cast<unsigned char*>(workspace);
    int parts = 1;
    while (parts < KNG_PARTS && static_cast<int64_t>(b) * 2 * parts <= TPK_COMPUTE_UNITS)
        parts *= 2;
    hipLaunchKernelGGL(knn_grid_build_kernel, dim3(static_cast<unsigned>(b) * parts), dim3(LG_THREADS), lds, stream, m, knn_per_cell(k), parts, layout,
                       support, w);
    const int64_t per_cloud = tpk_ceil_div(n, KNQ_QUERIES * (KNN_THREADS / TPK_WAVE));
    if (k <= KNQ_MAX_K && queries >= KNQ_LEAST && per_cloud * b <= 0x7fffffffLL)
    {
        auto* const kernel = k <= 8 ? &knn_grid_four_kernel<4> : &knn_grid_four_kernel<8>;
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(per_cloud * b)), dim3(KNN_THREADS), 0, stream, n, m, k, static_cast<unsigned>(per_cloud),
                           layout, query, w, dist2, idx);
        return tpk_launch_status();
    }
    hipLaunchKernelGGL(knn_grid_search_kernel, dim3(static_cast<unsigned>(blocks)), dim3(KNN_THREADS), 0, stream, queries, n, m, k, layout,
                       query, w, dist2, idx);
    return tpk_launch_status();
}

// The k nearest support points closer than `limit` (squared), for every query: search over
// curve-ordered cells where it applies and a workspace is given, otherwise all pairs.
int nearest_within(int b, int n_support, int m_query, int k, float limit, const float* support, const float* query,
                   int64_t* idx, float* dist2, void* workspace, size_t workspace_bytes, hipStream_t s)
{
    if (workspace)
    {
        const int st = tpk_grid_knn(b, m_query, n_support, k, limit, query, support, dist2, idx, workspace,
                                    workspace_bytes, s);
        if (st != TPK_ERR_UNSUPPORTED)
            return st;
    }
    if (k <= 4)
        return launch_knn<4>(b, m_query, n_support, k, limit, query, support, dist2, idx, s);
    if (k <= 8)
        return launch_knn<8>(b, m_query, n_support, k, limit, query, support, dist2, idx, s);
    if (k <= 16)
        return launch_knn<16>(b, m_query, n_support, k, limit, query, support, dist2, idx, s);
    return launch_knn<KNN_MAX_K>(b, m_query, n_support, k, limit, query, support, dist2, idx, s);
}

} // namespace

// (a list per lane over curve-ordered cells)
extern "C" size_t tpk_knn_workspace_bytes(int b, int n_support, int m_query)
{
    return tpk_grid_knn_workspace_bytes(b, m_query, n_support);
}

// (a wavefront per query over a grid in memory)
extern "C" size_t tpk_knn_grid_workspace_bytes(int b, int n_support, int m_query)
{
    return n_support > 0 ? knn_grid_workspace_bytes(b, n_support, m_query) : 0;
}

extern "C" int tpk_knn_f32(int b, int n_support, int m_query, int k, const float* support,
                           const float* query, int64_t* idx, float* dist2, void* workspace,
                           size_t workspace_bytes, void* stream)
{
    if (b < 0 || n_support < 0 || m_query < 0 || k < 0 || k > n_support)
        return TPK_ERR_INVALID_ARG; // (fewer support points than neighbours asked for)
    if (b == 0 || m_query == 0 || k == 0)
        return TPK_OK;
    if (!support || !query || !idx || !dist2)
        return TPK_ERR_INVALID_ARG;
    if (static_cast<int64_t>(n_support) * 3 > 0x7fffffffLL || static_cast<int64_t>(m_query) * 3 > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    const int cells = workspace ? knn_grid_cells(b, n_support, m_query, workspace_bytes) : 0; // of a grid in it
    if (k <= KNC_MAX_K && knn_in_lds(b, n_support, m_query, cells > 0))
        return launch_knn_cells(b, m_query, n_support, k, query, support, dist2, idx, tpk_stream(stream));
    if (k <= KNC_MAX_K && cells > 0)
        return launch_knn_grid(b, m_query, n_support, k, cells, query, support, dist2, idx, workspace, tpk_stream(stream));
    return nearest_within(b, n_support, m_query, k, __builtin_inff(), support, query, idx, dist2, workspace,
                          workspace_bytes, tpk_stream(stream));
}

// ---------------------------------------------------------------------------------------------
// Ball query with sorted neighbours: the nsample nearest support points closer than the radius,
// nearest first.  This is what the reference computes for CPU tensors with sort=True
// (cpu/src/neighbors.cpp:8-136 dense, :139-310 packed: nanoflann's radius search, which keeps
// a point when its squared distance is < radius * radius, sorted by distance and cut at max_num)
// and refuses for CUDA tensors (torch_points_kernels/torchpoints.py:152-153, :163-164).  Equal
// distances keep the lower index first (nanoflann sorts by distance only and leaves that open).
// Unused slots: dense - index of the nearest neighbour, or 0 when there is none, distance -1
// (neighbors.cpp:60-61, :88-105); packed - index -1, distance -1 (:248-275).
// ---------------------------------------------------------------------------------------------
namespace {

// Slots the search left empty read (limit, 0); they become the padding of the layout.
// Indices of found neighbours are raised by `add` (packed layout searched cloud by cloud: the
// position of the cloud's first support point).
__global__ __launch_bounds__(KNN_THREADS) void pad_sorted_kernel(int64_t slots, int nsample, float limit, bool packed,
                                                                 int64_t add, int64_t* __restrict__ idx,
                                                                 float* __restrict__ dist)
{
    const int64_t o = static_cast<int64_t>(blockIdx.x) * KNN_THREADS + threadIdx.x;
    if (o >= slots)
        return;
    const float d = dist[o];
    if (d < limit)
    {
        if (add != 0)
            idx[o] += add;
        return;
    }
    // The first slot of the row: the nearest neighbour, or the empty entry's 0 (also after this
    // kernel has padded it, in the dense layout).
    const int64_t token = packed ? -1 : idx[o - o % nsample];
    if (packed || o % nsample != 0)
        idx[o] = token;
    dist[o] = -1.0f;
}

int pad_sorted(int64_t rows, int nsample, float limit, bool packed, int64_t add, int64_t* idx, float* dist,
               hipStream_t s)
{
    const int64_t slots = rows * nsample;
    const int64_t blocks = tpk_ceil_div(slots, KNN_THREADS);
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(pad_sorted_kernel, dim3(static_cast<unsigned>(blocks)), dim3(KNN_THREADS), 0, s, slots, nsample,
                       limit, packed, add, idx, dist);
    return tpk_launch_status();
}

__device__ __forceinline__ int64_t first_not_below(const int64_t* __restrict__ a, int64_t n, int64_t v)
{
    int64_t lo = 0, hi = n;
    while (lo < hi)
    {
        const int64_t mid = (lo + hi) >> 1;
        if (a[mid] < v)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// Packed layout, all pairs: one lane owns one query.  The queries of a workgroup are consecutive,
// so they belong to a few clouds (the cloud ids are sorted); for each of those clouds its support
// points stream through LDS and the lanes of that cloud's queries scan them.
template <int K>
__global__ __launch_bounds__(KNN_THREADS) void nearest_packed_kernel(
    int64_t size_x, int64_t size_y, int nsample, int first, int count, float limit, const float* __restrict__ x,
    const float* __restrict__ y, const int64_t* __restrict__ batch_x, const int64_t* __restrict__ batch_y,
    int64_t* __restrict__ idx, float* __restrict__ dist)
{
    __shared__ float4 tile[KNN_TILE];

    const int tid = threadIdx.x;
    const int64_t q0 = static_cast<int64_t>(blockIdx.x) * KNN_THREADS;
    const int64_t q1 = tpk_min64(q0 + KNN_THREADS, size_y);
    const int64_t j = q0 + tid;
    const bool real = j < size_y;
    const int64_t jj = real ? j : size_y - 1;
    const float qx = y[jj * 3 + 0], qy = y[jj * 3 + 1], qz = y[jj * 3 + 2];
    const int64_t mine = batch_y[jj];
    NearestK<K> s;
    {
        const int64_t at = jj * nsample + first - 1;
        s.reset(first > 0, first > 0 ? dist[at] : 0.f, first > 0 ? static_cast<int>(idx[at]) : 0, !real, limit);
    }

    int64_t run_start = q0;
    while (run_start < q1) // the same runs for every lane of the workgroup
    {
        const int64_t c = batch_y[run_start];
        const int64_t run_end = tpk_min64(q1, q0 + first_not_below(batch_y + q0, q1 - q0, c + 1));
        const int64_t s0 = first_not_below(batch_x, size_x, c);
        const int64_t s1 = s0 + first_not_below(batch_x + s0, size_x - s0, c + 1);
        const bool in_run = real && mine == c;
        for (int64_t base = s0; base < s1; base += KNN_TILE)
        {
            const int cnt = static_cast<int>(tpk_min64(KNN_TILE, s1 - base));
            __syncthreads(); // the previous tile has been consumed by every wave
            for (int t = tid; t < cnt; t += KNN_THREADS)
            {
                const float* src = x + (base + t) * 3;
                tile[t] = make_float4(src[0], src[1], src[2], 0.f);
            }
            __syncthreads();
            if (in_run)
                scan_tile<K>(tile, cnt, static_cast<int>(base), qx, qy, qz, s);
        }
        run_start = run_end > run_start ? run_end : run_start + 1;
    }

    if (real)
    {
#pragma unroll
        for (int e = 0; e < K; ++e)
            if (e < count)
            {
                dist[j * nsample + first + e] = s.dist(e);
                idx[j * nsample + first + e] = s.index(e);
            }
    }
}

template <int K>
int launch_nearest_packed(int64_t size_x, int64_t size_y, int nsample, float limit, const float* x, const float* y,
                          const int64_t* batch_x, const int64_t* batch_y, int64_t* idx, float* dist, hipStream_t s)
{
    const int64_t blocks = tpk_ceil_div(size_y, KNN_THREADS);
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    for (int first = 0; first < nsample; first += K)
    {
        hipLaunchKernelGGL(nearest_packed_kernel<K>, dim3(static_cast<unsigned>(blocks)), dim3(KNN_THREADS), 0, s, size_x,
                           size_y, nsample, first, nsample - first < K ? nsample - first : K, limit, x, y, batch_x,
                           batch_y, idx, dist);
        const int st = tpk_launch_status();
        if (st != TPK_OK)
            return st;
    }
    return TPK_OK;
}

} // namespace

extern "C" size_t tpk_ball_query_sorted_dense_workspace_bytes(int b, int n, int m)
{
    // up to 64 neighbours: one wavefront per query over the ordered support points; more: the lists
    // of the k-nearest search, which orders both sets
    const size_t waves = tpk_grid_ball_sorted_workspace_bytes(b, n), lists = tpk_grid_knn_workspace_bytes(b, m, n);
    return waves > lists ? waves : lists;
}

extern "C" int tpk_ball_query_sorted_dense_f32(int b, int n, int m, float radius, int nsample, const float* new_xyz,
                                               const float* xyz, int64_t* idx, float* dist, void* workspace,
                                               size_t workspace_bytes, void* stream)
{
    if (b < 0 || n < 0 || m < 0 || nsample < 0)
        return TPK_ERR_INVALID_ARG;
    if (b == 0 || m == 0 || nsample == 0)
        return TPK_OK;
    if (!new_xyz || !idx || !dist || (n > 0 && !xyz))
        return TPK_ERR_INVALID_ARG;
    if (static_cast<int64_t>(n) * 3 > 0x7fffffffLL || static_cast<int64_t>(m) * 3 > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    hipStream_t s = tpk_stream(stream);
    const float limit = radius * radius; // fp32 product (cpu/src/neighbors.cpp:19)
    {
        // clouds that fit in LDS, up to 64 neighbours: buckets of cells built by every workgroup, no workspace
        const int cells = tpk_cells_ball_query_dense(b, n, m, radius, limit, nsample, true, new_xyz, xyz, idx, dist, s);
        if (cells != TPK_ERR_UNSUPPORTED)
            return cells; // (padding included)
    }
    if (workspace)
    {
        const int direct = tpk_grid_ball_sorted(b, m, n, nsample, limit, false, 0, new_xyz, xyz, dist, idx, workspace,
                                                workspace_bytes, s);
        if (direct != TPK_ERR_UNSUPPORTED)
            return direct; // (padding included)
    }
    const int st = nearest_within(b, n, m, nsample, limit, xyz, new_xyz, idx, dist, workspace, workspace_bytes, s);
    if (st != TPK_OK)
        return st;
    return pad_sorted(static_cast<int64_t>(b) * m, nsample, limit, false, 0, idx, dist, s);
}

namespace {

constexpr int NP_MAX_CLOUDS = 1024; // cloud ids served cloud by cloud; larger ids: all pairs in one launch

// ranges[c] / ranges[NP_MAX_CLOUDS + 1 + c]: position of the first support point / query with
// cloud id >= c, for c = 0 .. NP_MAX_CLOUDS.
__global__ __launch_bounds__(KNN_THREADS) void cloud_ranges_kernel(int64_t size_x, int64_t size_y,
                                                                   const int64_t* __restrict__ batch_x,
                                                                   const int64_t* __restrict__ batch_y,
                                                                   int64_t* __restrict__ ranges)
{
    const int c = blockIdx.x * KNN_THREADS + threadIdx.x;
    if (c > NP_MAX_CLOUDS)
        return;
    ranges[c] = first_not_below(batch_x, size_x, c);
    ranges[NP_MAX_CLOUDS + 1 + c] = first_not_below(batch_y, size_y, c);
}

int nearest_packed(int64_t size_x, int64_t size_y, int nsample, float limit, const float* x, const float* y,
                   const int64_t* batch_x, const int64_t* batch_y, int64_t* idx, float* dist, hipStream_t s)
{
    if (nsample <= 4)
        return launch_nearest_packed<4>(size_x, size_y, nsample, limit, x, y, batch_x, batch_y, idx, dist, s);
    if (nsample <= 8)
        return launch_nearest_packed<8>(size_x, size_y, nsample, limit, x, y, batch_x, batch_y, idx, dist, s);
    if (nsample <= 16)
        return launch_nearest_packed<16>(size_x, size_y, nsample, limit, x, y, batch_x, batch_y, idx, dist, s);
    return launch_nearest_packed<KNN_MAX_K>(size_x, size_y, nsample, limit, x, y, batch_x, batch_y, idx, dist, s);
}

constexpr size_t NP_RANGES_BYTES = (2 * (NP_MAX_CLOUDS + 1) * sizeof(int64_t) + 255) / 256 * 256;
constexpr int64_t NP_GRID_POINTS = 163840; // largest cloud the search over cells takes

} // namespace

// The workspace lets clouds of 512..163840 support points be searched over curve-ordered cells, one
// cloud after the other (up to 64 neighbours: one wavefront per query; more: the k-nearest lists,
// which also want 512 queries or more); the call then waits for the stream once, to read the
// clouds' ranges.
extern "C" size_t tpk_ball_query_sorted_partial_workspace_bytes(int64_t size_x, int64_t size_y)
{
    if (size_x < 512 || size_y < 1)
        return 0;
    const int most_x = static_cast<int>(tpk_min64(size_x, NP_GRID_POINTS));
    const size_t lists = tpk_grid_knn_workspace_bytes(1, static_cast<int>(tpk_min64(size_y, NP_GRID_POINTS)), most_x);
    const size_t waves = tpk_grid_ball_sorted_workspace_bytes(1, most_x);
    const size_t grid = waves > lists ? waves : lists;
    // (up to 64 neighbours the packed array is searched as a whole: no wait)
    const size_t table = tpk_table_ball_query_pays(size_x, size_y, true) ? tpk_table_ball_query_workspace_bytes(size_x, size_y, TPK_WAVE) : 0;
    const size_t bins = tpk_grid_ball_query_workspace_bytes(size_x, size_y, TPK_WAVE);
    const size_t cloudwise = grid ? NP_RANGES_BYTES + grid : 0;
    return std::max(std::max(table, bins), cloudwise);
}

extern "C" int tpk_ball_query_sorted_partial_f32(int64_t size_x, int64_t size_y, float radius, int nsample,
                                                 const float* x, const float* y, const int64_t* batch_x,
                                                 const int64_t* batch_y, int64_t* idx, float* dist, void* workspace,
                                                 size_t workspace_bytes, void* stream)
{
    if (size_x < 0 || size_y < 0 || nsample < 0)
        return TPK_ERR_INVALID_ARG;
    if (size_y == 0 || nsample == 0)
        return TPK_OK;
    if (!y || !batch_y || !idx || !dist || (size_x > 0 && (!x || !batch_x)))
        return TPK_ERR_INVALID_ARG;
    if (size_x > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    hipStream_t s = tpk_stream(stream);
    const float limit = radius * radius; // fp32 product (cpu/src/neighbors.cpp:153)
    const size_t wanted = tpk_ball_query_sorted_partial_workspace_bytes(size_x, size_y);
    if (!workspace || wanted == 0)
    {
        const int st = nearest_packed(size_x, size_y, nsample, limit, x, y, batch_x, batch_y, idx, dist, s);
        return st != TPK_OK ? st : pad_sorted(size_y, nsample, limit, true, 0, idx, dist, s);
    }
    if (workspace_bytes < wanted || (reinterpret_cast<uintptr_t>(workspace) & 255u))
        return TPK_ERR_WORKSPACE;
    if (nsample <= TPK_WAVE)
    {
        // The whole packed array at once - a hash table of cells, for few queries windows of consecutive rows and their bins -, the
        // rows of every query's cloud found on the device: no wait for the stream.
        int st = tpk_table_ball_query_partial(size_x, size_y, radius, limit, nsample, true, x, y, batch_x, batch_y, idx, dist, workspace,
                                              workspace_bytes, s);
        if (st == TPK_ERR_UNSUPPORTED)
            st = tpk_grid_ball_query_partial(size_x, size_y, radius, limit, nsample, true, x, y, batch_x, batch_y, idx, dist, workspace,
                                             workspace_bytes, s);
        if (st != TPK_ERR_UNSUPPORTED)
            return st;
    }

    // Where every cloud starts in both arrays.
    static_assert(NP_MAX_CLOUDS + 1 <= 5 * KNN_THREADS, "one thread per cloud id");
    int64_t* ranges_dev = static_cast<int64_t*>(workspace);
    hipLaunchKernelGGL(cloud_ranges_kernel, dim3(5), dim3(KNN_THREADS), 0, s, size_x, size_y, batch_x, batch_y, ranges_dev);
    int64_t ranges[2 * (NP_MAX_CLOUDS + 1)];
    static_assert(sizeof(ranges) <= TPK_READ_BACK_BYTES, "the cloud ranges fit the pinned buffer");
    const int read = tpk_read_back(ranges, ranges_dev, sizeof(ranges), s);
    if (read != TPK_OK)
        return read;
    const int64_t* rx = ranges;
    const int64_t* ry = ranges + NP_MAX_CLOUDS + 1;
    void* grid_ws = static_cast<char*>(workspace) + NP_RANGES_BYTES;
    const size_t grid_bytes = workspace_bytes - NP_RANGES_BYTES;

    // Queries q0..q1 (one cloud when `points` >= 0: its support points are s0 .. s0 + points).
    auto segment = [&](int64_t q0, int64_t q1, int64_t s0, int64_t points) -> int {
        if (q1 <= q0)
            return TPK_OK;
        const int64_t queries = q1 - q0;
        int64_t* idx_c = idx + q0 * nsample;
        float* dist_c = dist + q0 * nsample;
        int st = TPK_ERR_UNSUPPORTED;
        int64_t add = 0;
        if (points >= 0 && points <= NP_GRID_POINTS && queries <= 0x7fffffffLL)
        {
            // up to 64 neighbours: one wavefront per query over the cloud's ordered support points
            st = tpk_grid_ball_sorted(1, static_cast<int>(queries), static_cast<int>(points), nsample, limit, true, s0,
                                      y + q0 * 3, x + s0 * 3, dist_c, idx_c, grid_ws, grid_bytes, s);
            if (st != TPK_ERR_UNSUPPORTED)
                return st; // (padding included)
        }
        if (points >= 0 && queries <= NP_GRID_POINTS && points <= NP_GRID_POINTS &&
            tpk_grid_knn_workspace_bytes(1, static_cast<int>(queries), static_cast<int>(points)) != 0)
        {
            // search over cells; it numbers the support points from the cloud's first one
            st = tpk_grid_knn(1, static_cast<int>(queries), static_cast<int>(points), nsample, limit, y + q0 * 3,
                              x + s0 * 3, dist_c, idx_c, grid_ws, grid_bytes, s);
            add = s0;
        }
        if (st == TPK_ERR_UNSUPPORTED)
        {
            st = nearest_packed(size_x, queries, nsample, limit, x, y + q0 * 3, batch_x, batch_y + q0, idx_c, dist_c, s);
            add = 0;
        }
        return st != TPK_OK ? st : pad_sorted(queries, nsample, limit, true, add, idx_c, dist_c, s);
    };
    int st = segment(0, ry[0], 0, -1); // negative cloud ids, if any: all pairs
    for (int c = 0; c < NP_MAX_CLOUDS && st == TPK_OK; ++c)
        st = segment(ry[c], ry[c + 1], rx[c], rx[c + 1] - rx[c]);
    if (st == TPK_OK)
        st = segment(ry[NP_MAX_CLOUDS], size_y, 0, -1); // cloud ids of NP_MAX_CLOUDS and more: all pairs
    return st;
}
