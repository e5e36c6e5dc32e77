// Curve-ordered cells of point sets: the kernel that orders windows of at most CURVE_MAX_POINTS
// points along the curve (curve_order.h) and writes them out as cells of 64 records with their
// bounding boxes, for the searches that skip whole cells (nn_grid.hip) and for furthest point
// sampling of clouds too large for registers (fps.hip).
#pragma once

#include <algorithm>

#include "cloud_rows.h"
#include "curve_order.h"
#include "die_map.h"

namespace {

constexpr int NG_CELL = 64;           // points per cell = lanes of a wavefront
constexpr int NG_SORT_THREADS = 1024;
constexpr int CURVE_STAGED = 4096;    // records of a window's part that are put in order in LDS (64 KB)
constexpr int CURVE_PARTS = CURVE_MAX_POINTS / CURVE_STAGED; // parts of a window, at most
constexpr int NG_BOX = 2;             // float4 per cell: lowest and highest corner of its box
constexpr int NG_RUN_BOXES = 8;       // and of the boxes of its four runs of 16 points, which stand behind the boxes of all cells: the
                                      // searches read those of 64 cells at a time, a cell per lane (160 bytes apart, with the runs' boxes
                                      // between them, Chamfer's search lost a third of a wavefront's time on them)
constexpr int NG_CELL_BOXES = NG_BOX + NG_RUN_BOXES;

// A set of points to be ordered: `total` points in clouds of `cloud_points` consecutive points,
// every cloud cut into windows of `stride` consecutive points (the last window of a cloud may be
// shorter; a packed array of unequal clouds is one "cloud" whose windows hold whatever clouds
// lie there).  Every window gets stride / 64 (rounded up) cells of 64 records, in curve order; a record is (x, y, z, index inside the cloud), the
// padding records are infinitely far away with index 0x7FFFFFFF; a cell without points has an
// empty box (lo = +inf, hi = -inf).
struct PointSet
{
    const float* xyz;     // [total][3]
    const int64_t* group; // optional sorted cloud id per point (packed arrays), or nullptr
    int64_t total;
    int64_t cloud_points;
    int stride;
    float4* sorted;       // [windows][cells * 64]
    float4* boxes;        // [windows][cells][NG_BOX]: (lo.xyz, -), (hi.xyz, -) of the cells, then [windows][cells][NG_RUN_BOXES]: of their quarters; or nullptr
    int* bin_ends;        // optional [windows][CURVE_BINS]: end of every bin of the counting sort
    float4* grid;         // optional [windows][2]: origin and scale of the window's 64^3 grid
    int* wide_first;      // optional (with boxes) [windows][cells]: the cells of each of the window's parts (curve_parts()), those
                          // with much wider boxes than the part's average first - the cells whose queries take a search longest;
                          // the upper 16 bits of a part's first entry: how many of its cells are wide
    const int* only;      // optional [clouds]: a cloud whose word is 0 is left out (dense layout)
    const float4* records; // optional [total]: the points as (x, y, z, index) records to be read instead of xyz -
                           // an array that has been brought into a coarse order (coarse_order.h), whose records
                           // carry the numbers the points had before
};

__host__ __device__ inline int set_cells(const PointSet& s)
{
    return (s.stride + NG_CELL - 1) / NG_CELL;
}
__host__ __device__ inline int set_windows_per_cloud(const PointSet& s)
{
    return static_cast<int>((s.cloud_points + s.stride - 1) / s.stride);
}
__host__ __device__ inline int64_t set_windows(const PointSet& s)
{
    return s.total > 0 ? (s.total / s.cloud_points) * set_windows_per_cloud(s) : 0;
}

// A cell is wide when its box's squared diagonal exceeds this many times the average of its part of the window.  Chamfer forward of 32
// pairs of surfaces of 16384 points with 0.7 / 1 / 1.3 / 1.6 / 2 / 3 / 8: 136.5 / 135.2 / 134.7 / 135.8 / 138.1 / 143.1 / 144.8 us
// (none wide: 155); spheres with 1.3 and 3 113.3 and 120.7, clusters 222 and 228, even clouds 144.3 and 145.2.
constexpr float CURVE_WIDE_FACTOR = 1.3f;

// Orders part `part` of `parts` of a window of the set, by a workgroup of NG_SORT_THREADS; lds: curve_lds_bytes(), 16-byte aligned.
// The window's points are read once and stay in registers (16 per thread): bounding box, curve
// position of each point's cell of the 16^3 grid (a table in LDS), histogram and prefix sum over the
// 4096 bins, and then every thread takes a place in its points' bins (LDS integer atomics).
// Inside a bin (1/16 of the window's extent per axis) the order is that in which the atomics were
// served; it decides where a point sits inside its bin, never what a search over the cells returns.
//
// STAGED: the workgroup keeps the places of its part of the window's cells, puts their records in order in LDS and writes them and
// the boxes of their runs from there.  A record stored to its place by itself costs the compute unit's way to memory two clocks, as
// much as all the counting, and of the launch's windows there are fewer than compute units: every part counts the whole window and
// stores a share.  One window of 16384 points with boxes took 63000 clocks (18500 of them the stores, 20800 the boxes), a quarter of
// it takes 41000; the ordering of 64 of them 32.0 -> 22.9 us, Chamfer forward of 32 x 16384 points 164 -> 146, of one cloud 72 -> 62.
// Not STAGED (parts == 1; larger windows that are as many as compute units): the records go straight to their places, the boxes are
// formed from the records read back in order (one more trip to the L2 instead of random gathers of the coordinates).
template <bool STAGED>
__device__ __forceinline__ void curve_cells_part(const PointSet& set, int64_t window, int part, int parts, unsigned* lds)
{
    constexpr int PER = CURVE_MAX_POINTS / NG_SORT_THREADS; // points per thread
    unsigned* const bin_of_cell = lds;         // [CURVE_BINS] curve position of every cell of the 16^3 grid
    int* const bins = reinterpret_cast<int*>(bin_of_cell) + CURVE_BINS; // [CURVE_BINS]
    int* const run_boxes = bins + CURVE_BINS;  // [part's cells * 4][6] ordered ints: boxes of the runs of 16 records
    float4* const stage = reinterpret_cast<float4*>(run_boxes); // (STAGED) [part's cells * 64] the records, before run_boxes
    __shared__ int cloud_box[6];
    __shared__ int edge_bin[2], edge_start[2], edge_ends[2]; // the bins that hold the places before the part's first, and its last
    __shared__ unsigned edge_totals[NG_SORT_THREADS / TPK_WAVE];
    __shared__ int wave_totals[NG_SORT_THREADS / TPK_WAVE];
    __shared__ float wide_sums[NG_SORT_THREADS / TPK_WAVE];
    static_assert(CURVE_BINS % NG_SORT_THREADS == 0, "every thread scans the same number of bins");

    const int per_cloud = set_windows_per_cloud(set);
    const int64_t in_cloud = (window % per_cloud) * static_cast<int64_t>(set.stride);
    const int64_t start = (window / per_cloud) * set.cloud_points + in_cloud;
    const int n = static_cast<int>(tpk_min64(set.stride, set.cloud_points - in_cloud));
    const int cells = set_cells(set);
    // the cells of this part, and the places [place_lo, place_hi) of the points in them
    const int part_cells = (cells + parts - 1) / parts, cell_lo = min(part * part_cells, cells), cell_hi = min(cell_lo + part_cells, cells);
    const int place_lo = cell_lo * NG_CELL, place_hi = min(cell_hi * NG_CELL, n);
    const float* __restrict__ xyz = set.xyz + start * 3;
    const float4* __restrict__ records = set.records ? set.records + start : nullptr;
    const int64_t* __restrict__ group = set.group ? set.group + start : nullptr;
    float4* __restrict__ sorted = set.sorted + window * cells * NG_CELL;
    float4* __restrict__ boxes = set.boxes ? set.boxes + window * cells * NG_BOX : nullptr;
    float4* __restrict__ quarters = set.boxes ? set.boxes + set_windows(set) * cells * NG_BOX + window * cells * NG_RUN_BOXES : nullptr;
    const int tid = threadIdx.x;
    const int lane = tid & (TPK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / TPK_WAVE);

    // the points of this thread: tid, tid + 1024, ... (all loads issued before the first is used)
    float p[PER][3];
#pragma unroll
    for (int u = 0; u < PER; ++u)
    {
        const int k = min(tid + u * NG_SORT_THREADS, n - 1);
        if (records)
        {
            const float4 r = records[k];
            p[u][0] = r.x;
            p[u][1] = r.y;
            p[u][2] = r.z;
        }
        else
        {
#pragma unroll
            for (int a = 0; a < 3; ++a)
                p[u][a] = xyz[k * 3 + a];
        }
    }
    // (with cloud ids: how far a point's id lies above the window's first, cut at 7)
    int id_offset[PER];
    if (group)
    {
        const int64_t first_group = group[0];
#pragma unroll
        for (int u = 0; u < PER; ++u)
            id_offset[u] = static_cast<int>(tpk_min64(group[min(tid + u * NG_SORT_THREADS, n - 1)] - first_group, 7));
    }

    const int empty_lo = float_to_ordered_int(__builtin_inff());
    const int empty_hi = float_to_ordered_int(-__builtin_inff());
    if (tid < 6)
        cloud_box[tid] = tid < 3 ? empty_lo : empty_hi;
    if (tid < 2)
        edge_bin[tid] = -1;
    for (int i = tid; i < CURVE_BINS; i += NG_SORT_THREADS)
    {
        bins[i] = 0;
        bin_of_cell[i] = curve_bin_table.bin[i]; // (= curve_bin_of_cell(i & 15, (i >> 4) & 15, i >> 8))
    }
    __syncthreads();
    {
        // box of the window (only to quantise coordinates for the curve); the clamped loads repeat a real point
        float lo[3], hi[3];
#pragma unroll
        for (int a = 0; a < 3; ++a)
        {
            lo[a] = hi[a] = p[0][a];
#pragma unroll
            for (int u = 1; u < PER; ++u)
            {
                lo[a] = fminf(lo[a], p[u][a]);
                hi[a] = fmaxf(hi[a], p[u][a]);
            }
            const int wave_lo = wave_min_i32(float_to_ordered_int(lo[a]));
            const int wave_hi = wave_max_i32(float_to_ordered_int(hi[a]));
            if (lane == 0)
            {
                atomicMin(&cloud_box[a], wave_lo);
                atomicMax(&cloud_box[3 + a], wave_hi);
            }
        }
    }
    __syncthreads();

    // the bin of every point: position on the curve of its cell of the 16^3 grid (with cloud ids: the
    // first 7 distinct-id offsets come first, one id after the other, each in curve order; the rest together)
    int bin[PER];
    {
        const CurveGrid grid = curve_grid(cloud_box);
#pragma unroll
        for (int u = 0; u < PER; ++u)
        {
            bin[u] = -2; // no point
            if (u * NG_SORT_THREADS >= n) // (uniform over the workgroup: a short window has fewer rounds)
                continue;
            unsigned cell[3];
#pragma unroll
            for (int a = 0; a < 3; ++a)
                cell[a] = curve_grid_cell(p[u][a], grid.lo[a], grid.scale[a]);
            unsigned b = bin_of_cell[(cell[0] >> 2) | ((cell[1] >> 2) << 4) | ((cell[2] >> 2) << 8)];
            if (group)
            {
                b = (static_cast<unsigned>(id_offset[u]) << 9) | (b >> 3);
            }
            if (tid + u * NG_SORT_THREADS < n)
            {
                bin[u] = static_cast<int>(b);
                atomicAdd(&bins[b], 1);
            }
        }
    }
    __syncthreads();
    {
        // exclusive prefix sum over the bins: where every bin starts
        int count[CURVE_BINS / NG_SORT_THREADS];
        int sum = 0;
#pragma unroll
        for (int i = 0; i < CURVE_BINS / NG_SORT_THREADS; ++i)
        {
            count[i] = bins[tid * (CURVE_BINS / NG_SORT_THREADS) + i];
            sum += count[i];
        }
        const int before_in_wave = wave_exclusive_sum(sum);
        if (lane == TPK_WAVE - 1)
            wave_totals[wave] = before_in_wave + sum;
        __syncthreads();
        int run = before_in_wave;
        for (int w = 0; w < wave; ++w)
            run += wave_totals[w];
#pragma unroll
        for (int i = 0; i < CURVE_BINS / NG_SORT_THREADS; ++i)
        {
            const int b = tid * (CURVE_BINS / NG_SORT_THREADS) + i, end = run + count[i];
            bins[b] = run;
            run = end;
            if constexpr (!STAGED)
                continue;
#pragma unroll
            for (int edge = 0; edge < 2; ++edge)
            {
                const int at = edge == 0 ? place_lo : place_hi;
                if (end - count[i] < at && end >= at)
                {
                    edge_bin[edge] = b;
                    edge_start[edge] = end - count[i];
                    edge_ends[edge] = end;
                }
            }
            if (set.bin_ends && part == 0) // (the bin of a point is the leading 12 bits of its position on the curve: the cell
                set.bin_ends[window * CURVE_BINS + b] = end; // of the 16^3 grid it lies in, curve_bin_of_cell())
        }
    }
    __syncthreads();
    // every point takes the next place of its bin; its record goes straight there
    {
        // The part's bins.  A bin that also has places in the part before or behind is an edge of both; the places of its
        // points follow from their numbers, the same in both.
        const bool cut_lo = STAGED && edge_bin[0] >= 0 && edge_ends[0] > place_lo, cut_hi = STAGED && edge_bin[1] >= 0 && edge_ends[1] > place_hi;
        const int bin_lo = STAGED ? edge_bin[0] + 1 : 0, bin_hi = !STAGED ? CURVE_BINS : place_lo < place_hi ? edge_bin[1] + (cut_hi ? 0 : 1) : 0;
        int place[PER];
#pragma unroll
        for (int u = 0; u < PER; ++u)
            place[u] = bin[u] >= bin_lo && bin[u] < bin_hi ? atomicAdd(&bins[bin[u]], 1) : -1;
        if ((cut_lo || cut_hi) && place_lo < place_hi) // (uniform over the workgroup)
        {
            const int low = cut_lo ? edge_bin[0] : -1, high = cut_hi && edge_bin[1] != low ? edge_bin[1] : -1;
            bool any = false;
#pragma unroll
            for (int u = 0; u < PER; ++u)
                any = any || bin[u] == low || bin[u] == high;
            const bool some = __ballot(any) != 0; // (a bin holds a handful of points: few wavefronts have one)
            unsigned before = 0;                  // (points of the two edges in the halves of a word: at most 16384)
            if (some)
            {
                unsigned own = 0;
#pragma unroll
                for (int u = 0; u < PER; ++u)
                    own += (bin[u] == low ? 1u : 0u) + (bin[u] == high ? 0x10000u : 0u);
                before = static_cast<unsigned>(wave_exclusive_sum(static_cast<int>(own)));
                if (lane == TPK_WAVE - 1)
                    edge_totals[wave] = before + own;
            }
            else if (lane == 0)
                edge_totals[wave] = 0;
            __syncthreads();
            if (some)
            {
                for (int w = 0; w < wave; ++w)
                    before += edge_totals[w];
                const int start_lo = edge_start[0], start_hi = edge_start[1];
#pragma unroll
                for (int u = 0; u < PER; ++u)
                {
                    const bool in_low = bin[u] == low, in_high = bin[u] == high;
                    const int at = in_low ? start_lo + static_cast<int>(before & 0xFFFFu) : start_hi + static_cast<int>(before >> 16);
                    before += (in_low ? 1u : 0u) + (in_high ? 0x10000u : 0u);
                    if ((in_low || in_high) && at >= place_lo && at < place_hi)
                        place[u] = at;
                }
            }
        }
        // (records: the number a point had before the coarse order - read once more, the line is still near)
        int number[PER];
#pragma unroll
        for (int u = 0; u < PER; ++u)
            number[u] = static_cast<int>(in_cloud) + tid + u * NG_SORT_THREADS;
        if (records)
        {
#pragma unroll
            for (int u = 0; u < PER; ++u)
                if (place[u] >= 0)
                    number[u] = __float_as_int(records[tid + u * NG_SORT_THREADS].w);
        }
#pragma unroll
        for (int u = 0; u < PER; ++u)
            if (place[u] >= 0)
            {
                const float4 record = make_float4(p[u][0], p[u][1], p[u][2], __int_as_float(number[u]));
                if constexpr (STAGED)
                    stage[place[u] - place_lo] = record;
                else
                    sorted[place[u]] = record;
            }
    }
    const int padded = cell_hi * NG_CELL; // (of this part)
    {
        // records behind the last point: infinitely far away
        const float inf = __builtin_inff();
        for (int q = max(n, place_lo) + tid; q < padded; q += NG_SORT_THREADS)
        {
            const float4 record = make_float4(inf, inf, inf, __int_as_float(0x7FFFFFFF));
            if constexpr (STAGED)
                stage[q - place_lo] = record;
            else
                sorted[q] = record;
        }
    }
    int* const runs = STAGED ? reinterpret_cast<int*>(stage + part_cells * NG_CELL) : run_boxes;
    auto run_box_of = [&](int q, const float4& record) {
        const bool real = __float_as_int(record.w) != 0x7FFFFFFF;
        const float v[3] = {record.x, record.y, record.z};
        int lo[3], hi[3];
#pragma unroll
        for (int a = 0; a < 3; ++a)
        {
            const int ordered = float_to_ordered_int(v[a]);
            lo[a] = row_all_min_i32(real ? ordered : 0x7FFFFFFF);
            hi[a] = row_all_max_i32(real ? ordered : INT_MIN);
        }
        if ((lane & 15) == 0)
        {
            int* const run_box = runs + ((q - place_lo) / 16) * 6;
#pragma unroll
            for (int a = 0; a < 3; ++a)
            {
                run_box[a] = lo[a];
                run_box[3 + a] = hi[a];
            }
        }
    };
    // Every place is taken.  Not staged, the records have been stored, and the barrier
    // orders memory at workgroup scope, which is all the read-back below needs: the wavefronts of a workgroup share
    // one L1, which holds no older copy of these lines (a wider fence would write the whole L2 back: 20 us).
    __syncthreads();
    if constexpr (STAGED)
    {
        for (int q = place_lo + tid; q < padded; q += NG_SORT_THREADS)
        {
            const float4 record = stage[q - place_lo];
            sorted[q] = record;
            if (boxes) // boxes of the runs of 16 (DPP row reductions)
                run_box_of(q, record);
        }
    }
    else if (boxes)
    {
        // The records in order, as the other wavefronts stored them.
        constexpr int BATCH = 16; // (all records of a thread are requested before the first is used: one trip to the L2)
        for (int q0 = tid; q0 < padded; q0 += NG_SORT_THREADS * BATCH)
        {
            float4 rec[BATCH];
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
                rec[u] = sorted[min(q0 + u * NG_SORT_THREADS, padded - 1)];
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
                if (q0 + u * NG_SORT_THREADS < padded) // uniform over the wavefront: cells are whole
                    run_box_of(q0 + u * NG_SORT_THREADS, rec[u]);
        }
    }
    if (boxes)
    {
        // one thread per cell: the boxes of its four runs, and their union, to memory
        float diagonal2 = -1.f;
        __syncthreads();
        for (int c = cell_lo + tid; c < cell_hi; c += NG_SORT_THREADS)
        {
            // (an empty run keeps (INT_MAX, INT_MIN), which map to NaN patterns: written as (+inf, -inf))
            auto as_lo = [](int o) { return o == 0x7FFFFFFF ? __builtin_inff() : ordered_int_to_float(o); };
            auto as_hi = [](int o) { return o == INT_MIN ? -__builtin_inff() : ordered_int_to_float(o); };
            int lo[3] = {0x7FFFFFFF, 0x7FFFFFFF, 0x7FFFFFFF}, hi[3] = {INT_MIN, INT_MIN, INT_MIN};
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                const int* const run_box = runs + ((c - cell_lo) * 4 + r) * 6;
                quarters[c * NG_RUN_BOXES + r * 2 + 0] = make_float4(as_lo(run_box[0]), as_lo(run_box[1]), as_lo(run_box[2]), 0.f);
                quarters[c * NG_RUN_BOXES + r * 2 + 1] = make_float4(as_hi(run_box[3]), as_hi(run_box[4]), as_hi(run_box[5]), 0.f);
#pragma unroll
                for (int a = 0; a < 3; ++a)
                {
                    lo[a] = min(lo[a], run_box[a]);
                    hi[a] = max(hi[a], run_box[3 + a]);
                }
            }
            boxes[c * NG_BOX + 0] = make_float4(as_lo(lo[0]), as_lo(lo[1]), as_lo(lo[2]), 0.f);
            boxes[c * NG_BOX + 1] = make_float4(as_hi(hi[0]), as_hi(hi[1]), as_hi(hi[2]), 0.f);
            if (c == cell_lo + tid && lo[0] != 0x7FFFFFFF) // (a cell that holds points: the squared diagonal of its box)
            {
                const float dx = as_hi(hi[0]) - as_lo(lo[0]), dy = as_hi(hi[1]) - as_lo(lo[1]), dz = as_hi(hi[2]) - as_lo(lo[2]);
                diagonal2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
            }
        }
        if (set.wide_first) // (cells <= 256: one cell per thread of the first four wavefronts)
        {
            // the average over the cells that hold points, then the wide cells first, both groups in curve order
            const bool holds = diagonal2 >= 0.f;
            const float wave_sum = wave_sum_f32(holds ? diagonal2 : 0.f);
            const int wave_count = __builtin_popcountll(__ballot(holds));
            if (lane == 0)
            {
                wide_sums[wave] = wave_sum;
                wave_totals[wave] = wave_count;
            }
            __syncthreads();
            float sum = 0.f;
            int count = 0;
            for (int w = 0; w < NG_SORT_THREADS / TPK_WAVE; ++w)
            {
                sum += wide_sums[w];
                count += wave_totals[w];
            }
            const bool wide = holds && diagonal2 * count > CURVE_WIDE_FACTOR * sum;
            const unsigned long long wide_lanes = __ballot(wide);
            __syncthreads();
            if (lane == 0)
                wave_totals[wave] = __builtin_popcountll(wide_lanes);
            __syncthreads();
            int before = static_cast<int>(tpk_prefix_count(wide_lanes)), all_wide = 0;
            for (int w = 0; w < NG_SORT_THREADS / TPK_WAVE; ++w)
            {
                before += w < wave ? wave_totals[w] : 0;
                all_wide += wave_totals[w];
            }
            if (tid < cell_hi - cell_lo)
            {
                const int at = wide ? before : all_wide + tid - before;
                set.wide_first[window * cells + cell_lo + at] = (cell_lo + tid) | (at == 0 ? all_wide << 16 : 0);
            }
        }
    }
    if constexpr (!STAGED)
        if (set.bin_ends) // bins[i] is the end of bin i on the curve: every place is taken
            for (int i = tid; i < CURVE_BINS; i += NG_SORT_THREADS)
                set.bin_ends[window * CURVE_BINS + i] = bins[i];
    if (set.bin_ends && part == 0 && tid == 0)
    {
        const CurveGrid grid = curve_grid(cloud_box);
        set.grid[window * 2 + 0] = make_float4(grid.lo[0], grid.lo[1], grid.lo[2], 0.f);
        set.grid[window * 2 + 1] = make_float4(grid.scale[0], grid.scale[1], grid.scale[2], 0.f);
    }
}

// The ordering of two sets: the first windows_a windows are those of set_a, the rest set_b.
// `zero_word` (optional) is cleared by the first block: a counter used by the kernel that follows.
template <bool STAGED>
__global__ __launch_bounds__(NG_SORT_THREADS) void curve_cells_kernel(PointSet set_a, PointSet set_b,
                                                                      int windows_a, int windows, int parts, int* zero_word,
                                                                      CloudRows rows_job)
{
    extern __shared__ unsigned curve_lds[];
    const unsigned ordering = parts_grid(static_cast<unsigned>(windows), static_cast<unsigned>(parts));
    if (blockIdx.x >= ordering)
    {
        cloud_rows_job(rows_job, static_cast<int64_t>(blockIdx.x - ordering) * (NG_SORT_THREADS / TPK_WAVE) + threadIdx.x / TPK_WAVE,
                       threadIdx.x & (TPK_WAVE - 1));
        return;
    }
    // (The workgroups of a window run on one die, which reads the window once: 14900 -> 6000 clocks for the loads.  With blocks
    // instead of windows dealt to the dies that held for some grids only: Chamfer forward of 1 x 5000 points 53.1 -> 51.4 us, 1 x 12000
    // 66.4 -> 64.6, 3 x 5000 53.3 -> 52.1, 2 x 16384 90.0 -> 91.5.)
    const PartTask task = part_task(blockIdx.x, static_cast<unsigned>(windows), static_cast<unsigned>(parts));
    const int block = static_cast<int>(task.item);
    if (zero_word && blockIdx.x == 0 && threadIdx.x == 0)
        *zero_word = 0;
    if (block >= windows)
        return;
    const bool first_set = block < windows_a;
    const PointSet set = first_set ? set_a : set_b;
    const int64_t window = first_set ? block : block - windows_a;
    if (set.only && set.only[window / set_windows_per_cloud(set)] == 0)
        return;
    curve_cells_part<STAGED>(set, window, static_cast<int>(task.part), parts, curve_lds);
}

// Bytes of LDS for a part of `part_cells` cells.
inline size_t curve_lds_bytes(int64_t part_cells, bool staged)
{
    return (2 * static_cast<size_t>(CURVE_BINS) + 24 * static_cast<size_t>(part_cells)) * sizeof(unsigned) +
           (staged ? static_cast<size_t>(part_cells) * NG_CELL * sizeof(float4) : 0);
}

// Squared distance between two boxes / a point and a box (0 when they touch or overlap).
__device__ __forceinline__ float box_box_dist2(float4 alo, float4 ahi, float4 blo, float4 bhi)
{
    const float dx = fmaxf(fmaxf(blo.x - ahi.x, alo.x - bhi.x), 0.f);
    const float dy = fmaxf(fmaxf(blo.y - ahi.y, alo.y - bhi.y), 0.f);
    const float dz = fmaxf(fmaxf(blo.z - ahi.z, alo.z - bhi.z), 0.f);
    return __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
}
__device__ __forceinline__ float point_box_dist2(float x, float y, float z, float4 blo, float4 bhi)
{
    const float dx = fmaxf(fmaxf(blo.x - x, x - bhi.x), 0.f);
    const float dy = fmaxf(fmaxf(blo.y - y, y - bhi.y), 0.f);
    const float dz = fmaxf(fmaxf(blo.z - z, z - bhi.z), 0.f);
    return __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
}

// (of sets that hold points)
int largest_window(const PointSet& a, const PointSet& c)
{
    return std::max(a.total > 0 ? a.stride : 1, c.total > 0 ? c.stride : 1);
}

// Parts that the windows of a launch are cut into: such that a part's records fit in LDS, where the windows then still have a compute
// unit per part; otherwise one.
int curve_parts(const PointSet& a, const PointSet& c)
{
    const int64_t parts = tpk_ceil_div(largest_window(a, c), CURVE_STAGED);
    return (set_windows(a) + set_windows(c)) * parts <= TPK_COMPUTE_UNITS ? static_cast<int>(parts) : 1;
}

int launch_curve_cells(const PointSet& a, const PointSet& c, int* zero_word, hipStream_t s,
                       const CloudRows& rows_job = CloudRows{nullptr, nullptr, 0, 0, nullptr})
{
    const int largest = largest_window(a, c);
    if (largest > CURVE_MAX_POINTS)
        return TPK_ERR_UNSUPPORTED; // (a thread holds 16 points of a window: windows of at most 16384 points)
    const int64_t windows_a = set_windows(a), windows_c = set_windows(c);
    const int64_t row_groups = tpk_ceil_div(rows_job.size_y, NG_SORT_THREADS);
    if ((windows_a + windows_c + DIES) * CURVE_PARTS + row_groups > 0x7fffffffLL || windows_a + windows_c >= 1LL << 29)
        return TPK_ERR_UNSUPPORTED;
    const int parts = curve_parts(a, c);
    const int64_t part_cells = tpk_ceil_div(tpk_ceil_div(largest, NG_CELL), parts);
    const bool staged = part_cells * NG_CELL <= CURVE_STAGED;
    const size_t lds = curve_lds_bytes(part_cells, staged);
    const auto kernel = staged ? curve_cells_kernel<true> : curve_cells_kernel<false>;
    const int allowed = tpk_allow_lds(reinterpret_cast<const void*>(kernel), lds);
    if (allowed != TPK_OK)
        return allowed;
    hipLaunchKernelGGL(kernel, dim3(parts_grid(static_cast<unsigned>(windows_a + windows_c), static_cast<unsigned>(parts)) + static_cast<unsigned>(row_groups)),
                       dim3(NG_SORT_THREADS), lds, s, a, c, static_cast<int>(windows_a),
                       static_cast<int>(windows_a + windows_c), parts, zero_word, rows_job);
    return tpk_launch_status();
}

} // namespace
