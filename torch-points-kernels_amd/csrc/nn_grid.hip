// Nearest-neighbour search over clouds cut into spatially compact cells.
//
// The all-pairs scans (chamfer.hip, three_nn.hip) test every query against every candidate.
// Here both clouds are first ordered along a Hilbert curve (curve_order.h) and cut into cells
// of 64 consecutive points, each with its bounding box.  A wavefront then serves the 64
// queries of one cell: it measures the distance from its cell's box to every candidate cell's
// box (one lane per candidate cell), scans the nearest candidate cell to get a first answer,
// and afterwards scans only candidate cells whose box is not further away than the worst
// current answer of its lanes.  A skipped cell cannot hold a nearer point, nor one at equal
// distance: the box distance is compared with a relative margin of 2e-6, several times the fp32
// rounding error of either side.  Distances of the pairs that are evaluated use the same
// operations in the same order as the all-pairs kernels, so values are bit-identical.
//
// The candidates are visited in curve order, not index order, so "the lowest index among equal
// distances" - what a serial first-strictly-smaller scan returns - is enforced explicitly: the
// scan keeps the minimum and the first group of 8 candidates that reached it, and flags a lane
// when another group reaches the same value; flagged lanes (duplicated points, lattices) take
// an extra pass that collects the lowest index among all candidates at that distance.  Chamfer's
// scan runs on the matrix cores and asks for that pass where two candidates are too close to tell.
//
// Workspace per cloud: 16 bytes per point (x, y, z, original index) padded to whole cells, and
// 160 bytes per cell (its box and those of its four runs of 16 points).  The curve ordering works
// in LDS on at most 16384 points: a larger cloud (up to 163840 points) is ordered in windows of
// 16384 consecutive points, which the search sees as more - and wider - cells of the same cloud.
#include "curve_cells.h"

#include <algorithm>
#include <cmath>
#include "ball_scan.h"
#include "nn_grid.h"
#include "topk.h"

namespace {

constexpr int NG_MAX_CELLS = 2560;           // candidate cells per cloud (their box distances sit in LDS)
constexpr int NG_WINDOW = CURVE_MAX_POINTS;  // larger clouds are ordered in windows of this many points
constexpr int NG_SCAN_THREADS = 256;         // 4 wavefronts, each searching on its own
constexpr float NG_MARGIN = 0.999998f;
constexpr int NG_CHUNK = 8;

// Box of the 64 queries of a wavefront (one query per lane; a padding lane - index 0x7FFFFFFF - holds none),
// the same value in every lane.  The ordering kernel forms no boxes for a set that is only queried.
__device__ __forceinline__ void query_box(float qx, float qy, float qz, bool real, float4& lo, float4& hi)
{
    const float v[3] = {qx, qy, qz};
    float l[3], h[3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
    {
        const int ordered = float_to_ordered_int(v[a]);
        l[a] = ordered_int_to_float(wave_min_i32(real ? ordered : float_to_ordered_int(__builtin_inff())));
        h[a] = ordered_int_to_float(wave_max_i32(real ? ordered : float_to_ordered_int(-__builtin_inff())));
    }
    lo = make_float4(l[0], l[1], l[2], 0.f);
    hi = make_float4(h[0], h[1], h[2], 0.f);
}

// State of one lane's nearest-neighbour search.
struct Nearest
{
    float best; // smallest distance so far
    int chunk;  // first group of NG_CHUNK candidates (position / NG_CHUNK on the curve) that reached it
    bool tie;   // another group reached the same value
};

// Scans candidate cell `cell` for the 64 queries of the wavefront.  `stage` is the wavefront's
// own 64-entry LDS buffer, through which every lane sees every candidate (broadcast reads).
__device__ __forceinline__ void scan_cell(const float4* __restrict__ cand, const float4* __restrict__ runs,
                                          int cell, float4* stage, int lane, float qx, float qy, float qz,
                                          Nearest& s TPK_WORK_PARAM)
{
    stage[lane] = cand[cell * NG_CELL + lane];
    // (the boxes of the cell's four runs are requested together with its candidates: one wait, not five)
    float4 quarter[NG_RUN_BOXES];
#pragma unroll
    for (int i = 0; i < NG_RUN_BOXES; ++i)
        quarter[i] = runs[cell * NG_RUN_BOXES + i];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); // LDS serves a wavefront's requests in order
#pragma unroll
    for (int run = 0; run < NG_CELL / (2 * NG_CHUNK); ++run)
    {
        // a run of 16 candidates whose box no lane's answer reaches is passed over
        const float lb = point_box_dist2(qx, qy, qz, quarter[2 * run], quarter[2 * run + 1]);
        if (__ballot(lb * NG_MARGIN <= s.best) == 0)
            continue;
#pragma unroll
        for (int half = 0; half < 2; ++half)
        {
            const int ch = 2 * run + half;
            float mn = 0.f;
#pragma unroll
            for (int c = 0; c < NG_CHUNK; ++c)
            {
                const float4 p = stage[ch * NG_CHUNK + c];
                // Operand order of the reference: (scanned - query), squares summed x, y, z.
                const float d = tpk_dist2(p.x, p.y, p.z, qx, qy, qz);
                mn = c == 0 ? d : fminf(mn, d);
            }
            TPK_WORK_ADD(NG_CHUNK);
            const bool better = mn < s.best;
            const bool equal = mn == s.best;
            s.tie = better ? false : (s.tie || equal);
            s.chunk = better ? cell * (NG_CELL / NG_CHUNK) + ch : s.chunk;
            s.best = better ? mn : s.best;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The same for a cell that only a few queries of the wavefront still ask for (an outlier among the
// queries keeps admitting cells that the other 63 have long turned down): one query at a time, the
// 64 candidates of the cell side by side in the lanes.  `want`: the lanes whose queries ask.
// A minimum reached in the cell by several groups of NG_CHUNK candidates, or equal to the query's
// answer so far, sets the tie flag exactly as the scan above would.
constexpr int NG_DEAL = 8;   // windows whose cells are dealt out together, wide cells first
constexpr int NG_FEW = 8; // (the scan above costs about as much as 14 queries served this way; 16: the same time, 24: slower)
__device__ __forceinline__ void scan_cell_few(const float4* __restrict__ cand, int cell, unsigned long long want,
                                              int lane, float qx, float qy, float qz, Nearest& s TPK_WORK_PARAM)
{
    const float4 p = cand[cell * NG_CELL + lane];
    while (want != 0)
    {
        const int q = __builtin_ctzll(want);
        want &= want - 1;
        TPK_WORK_ADD(1);
        const float ux = tpk_read_lane(qx, q), uy = tpk_read_lane(qy, q), uz = tpk_read_lane(qz, q);
        const float d = tpk_dist2(p.x, p.y, p.z, ux, uy, uz); // (a padding candidate lies at infinity)
        // distances are >= +0: their bit patterns order like unsigned integers (a NaN of either sign sorts above infinity; what the
        // device itself makes of 0 / 0 or infinity minus infinity has the sign set)
        const float mn = __int_as_float(static_cast<int>(wave_min_u32(static_cast<unsigned>(__float_as_int(d)))));
        const unsigned long long at = __ballot(d == mn);
        if (at == 0)
            continue; // nothing but NaN
        const int first = __builtin_ctzll(at);
        const bool several = (at & ~(0xFFull << (first & ~(NG_CHUNK - 1)))) != 0;
        if (lane == q)
        {
            const bool better = mn < s.best;
            const bool equal = mn == s.best;
            s.tie = better ? several : (s.tie || equal);
            s.chunk = better ? cell * (NG_CELL / NG_CHUNK) + first / NG_CHUNK : s.chunk;
            s.best = better ? mn : s.best;
        }
    }
}

// ---- Chamfer's scan on the matrix cores --------------------------------------------------
// |p - q|^2 = |p|^2 - 2 p.q + |q|^2 is a product over 16 slots once every number is given as two halves, so one
// v_mfma_f32_32x32x16_f16 forms 32 x 32 distances.  They are not the distances the search returns: they say which
// eight candidates hold a query's answer, and those are evaluated as ever.  Coordinates are taken relative to the centre of
// the queries' box and scaled by a power of two; in these units everything the search needs lies within 1024 of the
// centre along every axis, and candidates further off than 16384 count as that far away.
//
// A candidate's row of the product: x, y (high halves), x, y (low), z, |p|^2 (high), z, |p|^2 (low), then x, y (high), x, y (low), z, |p|^2
// (high), 2^14, 2^14; against a query's -2x, -2y (high, twice), (-2z, 2^14) (high, twice), -2x, -2y (low, twice), (-2z, 0) (low), |q|^2 (high, low).
// The squares are kept divided by 2^14.
//
// The error of a product, in units of 2^-20 (|p| + |q|)^2: two halves hold 22 bits, which costs 2 p.q 0.38 and the squares, formed in
// float, 0.44; the frame 0.13; the sum of 16 products 0.88, 14 x 2^-24 of the sum of their magnitudes.  (Terms are cut off at about 2^-24 of the
// largest: random sums are off by up to 2.3 of these 14, sums made for it - one large term, the others just below the cut, of both signs - by 9.)
// As (|p| + |q|)^2 <= 4.4 |q|^2 + 11 |p - q|^2, that is 1.82 x 2^-20 times it: below MX_ERROR of |q|^2 and, with 0.4 for the two bits that a smallest
// product gives up for its place and 0.3 for the rounding of the distances themselves, MX_ERROR_NEAR of |p - q|^2.  Where a low half is below the
// normal range the products are off by less than 2^-8 more (2^-25 of a slot, against at most 2 x 1100 or 2^14); 2^-4 is allowed for it.
// What the unit's sums are off by, and that halves below the normal range count, is not documented but measured, and tested on the device
// (tpk_matrix_product, counting build); the search is run on the host with sums that far off.
//
// A query for which the eight and some other candidate are closer together than that (of 32 x 16384 points one in 3200 of even clouds, one in
// 1200 on a sphere) goes to the pass for equal minima; where many of a wavefront's do, the exact scan above answers
// them, a search of its own that starts with what is known: serving 64 of them one at a time took 2.8 times as long on clouds with outliers.
//
// What bounds it: the issue of vector instructions, ~105 for 64 x 64 pairs (22 to form the halves, 60 for the minima) where the
// exact scan takes ten per candidate.  32 x 16384 points, forward, with the ordering: a noisy sphere 116 -> 80 us (surfaces, with what else a
// pass does 122 -> 65 for the search alone), uniform 140 -> 98, eight clusters 182 -> 94; 2 x 60000 uniform 154 -> 101.
// Taken back: minima of four candidates (24 more instructions per scan, 12 % slower), whole wavefronts by the exact scan where many
// queries are left over (laser scans 30 % slower than without the matrix cores).
typedef _Float16 half2_t __attribute__((vector_size(4)));
typedef _Float16 half8_t __attribute__((vector_size(16)));
typedef float float16_t __attribute__((vector_size(64)));
typedef unsigned uint4_t __attribute__((vector_size(16)));

constexpr float MX_FAR = 16384.f;          // 2^14: candidates are clamped to this; also the factor |p|^2 and |q|^2 are kept divided by
constexpr float MX_LIMIT = 134217728.f;    // 2^27: a squared distance that no clamped candidate can have
constexpr float MX_NEAR = 8.f;             // largest distance of the first cell, in extents of its box and the queries'
constexpr float MX_ERROR = 0x1p-17f;       // of |q|^2, 8 x 2^-20 (above)
constexpr float MX_ERROR_NEAR = 0x1.8p-16f; // and of a product, 24 x 2^-20
// Who answers the queries that the products cannot: the pass for equal minima costs a query a look at all boxes and at the cells within its
// reach, the exact scan costs a wavefront its whole search again.  us, before the matrix cores / products with an exact scan of more than 20 queries,
// whatever the search was like / as here.
// - Left to the exact scan at once: more than MX_MANY queries for which two groups of the first cell are within MX_CLOSE errors of nothing, or too
//   close to each other.  Points with twins a few units in the last place away 32 x 16384 147 / 176 / 152, points on a line 8 x 16384 144 / 171 / 162.
// - Given up behind the overlapping cells: more than MX_MOST too close to each other, and those not blind, that is, with a smallest product above its
//   error (the blind go on: what they learn shortens the exact scan).  Twins in other windows 2 x 60000 170 / 244 / 188.
// - One by one, up to MX_PASS, and more of them where a query has MX_SCANS scans of the search to itself and half are not blind: wide cells, whose
//   search is long and whose queries are few and far apart.  Laser scans 2 x 60000 868 / 944 / 815, 2 x 100000 2110 / 1990 / 1960.  (All such
//   wavefronts, blind or not: 670 and 1640, but clouds with outliers 2 x 60000 2900 instead of 2690.)
// The reach of those left over ends at the best of their eight: clouds with outliers 32 x 4096 270 / 232 / 213, scaled point by point by e^0 .. e^-12
// 8 x 16384 890 / 960 / 933.  Still behind the search without products: these, twins, lines, and outliers in small calls (8 x 8192 on 2048 327 / 390 / 387).
// Taken back: giving up inside the overlapping cells, after 8, 16, 32 .. scans (outliers and lines 5 to 10 % faster, every call 3 % slower, by what each
// scan has to keep) or between groups of 64 cells (a line 2 x 60000 480 -> 439, outliers 2 x 16384 695 -> 623, every call 1 % slower).
constexpr float MX_CLOSE = 16.f;
constexpr int MX_MANY = 8;                 // (of 64; 16: twins 156, line 171)
constexpr int MX_MOST = 32;
constexpr int MX_SCANS = 8;                // (4: outliers 8 x 16384 1027 instead of 910)
// (12: laser scans of 32 x 4096 106 us against 91, e^-4 2 x 60000 1470 against 930; 32: a tail of slow wavefronts.  Not less in wavefronts that share a
// cell: halves with 10, laser scans of 2 x 16384 223 against 151, 8 x 8192 on 2048 144 against 93.)
constexpr int MX_PASS = 20;

// Two halves that add up to v: the rounded value, and what is left of it, rounded.
// (`minus_one` as a variable: the compiler then takes three instructions for a pair, v_fma_mix among them, instead of nine)
__device__ __forceinline__ void split_half(float a, float b, float minus_one, half2_t& high, half2_t& low)
{
    high = half2_t{static_cast<_Float16>(a), static_cast<_Float16>(b)};
    low = half2_t{static_cast<_Float16>(__builtin_fmaf(static_cast<float>(high[0]), minus_one, a)),
                  static_cast<_Float16>(__builtin_fmaf(static_cast<float>(high[1]), minus_one, b))};
}

// Operands of two tiles of 32 points, one point per lane: lanes 0 .. 31 of a tile hold slots 0 .. 7 of its points, the others slots 8 .. 15.
__device__ __forceinline__ void tile_operands(const half2_t (&first)[4], const half2_t (&second)[4], half8_t (&tile)[2])
{
    uint4_t t[2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        const auto swapped = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, first[i]),
                                                              __builtin_bit_cast(unsigned, second[i]), false, false);
        t[0][i] = swapped[0];
        t[1][i] = swapped[1];
    }
    tile[0] = __builtin_bit_cast(half8_t, t[0]);
    tile[1] = __builtin_bit_cast(half8_t, t[1]);
}

// v of the two tiles of 32 queries as the products leave them (lane l: query l % 32, the candidates of half l / 32) -> of
// query `lane` (query 32 j + i stands in lane 32 j + i), of either half of the candidates.
__device__ __forceinline__ void by_query(int tile0, int tile1, int& half0, int& half1)
{
    const auto swapped = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(tile0), static_cast<unsigned>(tile1), false, false);
    half0 = static_cast<int>(swapped[0]);
    half1 = static_cast<int>(swapped[1]);
}

// What a lane knows of one query and half of the candidates: the smallest and the second smallest of the minima of eight
// candidates (bit patterns; a negative one stands for a distance below the error), the place of the eight in their
// cell in the two lowest bits, and the smallest one's cell.
struct MatrixNearest
{
    int m1, m2, cell;
};

__device__ __forceinline__ void take_products(const float16_t& d, int tile, MatrixNearest& s)
{
#pragma unroll
    for (int q = 0; q < 2; ++q)
    {
        int eight = __float_as_int(d[8 * q]);
#pragma unroll
        for (int r = 1; r < 8; ++r)
            eight = min(eight, __float_as_int(d[8 * q + r]));
        const int v = (eight & ~3) | (tile * 2 + q);
        s.m2 = __float_as_int(__builtin_amdgcn_fmed3f(__int_as_float(s.m1), __int_as_float(s.m2), __int_as_float(v)));
        s.m1 = min(s.m1, v);
    }
    // (the second smallest are not looked at before the search ends: without this the compiler keeps what they follow from in
    // registers beyond the scan, 32 of them)
    asm volatile("" : "+v"(s.m2));
}

#ifdef TPK_COUNT_WORK
// One product per wavefront, for a test of what the bound above assumes of the unit.
__global__ __launch_bounds__(TPK_WAVE) void matrix_product_kernel(const uint4* __restrict__ a, const uint4* __restrict__ b, float* __restrict__ d)
{
    const int lane = threadIdx.x;
    const int64_t at = static_cast<int64_t>(blockIdx.x) * TPK_WAVE + lane;
    const float16_t sums = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a[at]), __builtin_bit_cast(half8_t, b[at]), float16_t{}, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; ++r)
        d[(static_cast<int64_t>(blockIdx.x) * 32 + r % 4 + 8 * (r / 4) + 4 * (lane / 32)) * 32 + lane % 32] = sums[r];
}
#endif

// Units of a wavefront's search: point * scale + offset.
struct MatrixFrame
{
    float scale, ox, oy, oz, minus_one;
};

// (`want`: the queries that ask for the cell; a tile of 32 queries, neighbours on the curve, of which none does is left out)
__device__ __forceinline__ void matrix_scan(const float4* __restrict__ cand, int cell, unsigned long long want, int lane, const MatrixFrame& f,
                                            const half8_t (&queries)[2], MatrixNearest (&s)[2] TPK_PRODUCTS_PARAM)
{
    const float4 p = cand[cell * NG_CELL + lane];
    // (a padding candidate, infinitely far away, and one that is not a number count as far away)
    const float x = __builtin_amdgcn_fmed3f(__builtin_fmaf(p.x, f.scale, f.ox), -MX_FAR, MX_FAR);
    const float y = __builtin_amdgcn_fmed3f(__builtin_fmaf(p.y, f.scale, f.oy), -MX_FAR, MX_FAR);
    const float z = __builtin_amdgcn_fmed3f(__builtin_fmaf(p.z, f.scale, f.oz), -MX_FAR, MX_FAR);
    const float square = __builtin_fmaf(x, x, __builtin_fmaf(y, y, z * z)) * (1.f / MX_FAR);
    half2_t xy_high, xy_low, zs_high, zs_low;
    split_half(x, y, f.minus_one, xy_high, xy_low);
    split_half(z, square, f.minus_one, zs_high, zs_low);
    const half2_t scale_slots = half2_t{static_cast<_Float16>(MX_FAR), static_cast<_Float16>(MX_FAR)};
    half8_t tiles[2];
    tile_operands({xy_high, xy_low, zs_high, zs_low}, {xy_high, xy_low, zs_high, scale_slots}, tiles);
#pragma unroll
    for (int j = 0; j < 2; ++j)
    {
        if (static_cast<unsigned>(want >> (32 * j)) == 0)
            continue;
        TPK_PRODUCTS_ADD(32); // (32 queries and 64 candidates, counted by 64 lanes)
        const int before = s[j].m1;
#pragma unroll
        for (int i = 0; i < 2; ++i)
        {
            const float16_t d = __builtin_amdgcn_mfma_f32_32x32x16_f16(tiles[i], queries[j], float16_t{}, 0, 0, 0);
            take_products(d, i, s[j]);
        }
        s[j].cell = s[j].m1 != before ? cell : s[j].cell;
        __builtin_amdgcn_sched_barrier(0);
    }
}

// One wavefront = the 64 queries of one cell, or a half or a quarter of them.  Logical wavefront number (after the
// die-local block mapping) = cloud * (cells1 + cells2) + cell, times the parts; the cells of cloud 1 query cloud 2 and
// write dist1 / idx1, those of cloud 2 the other way round.
__global__ __launch_bounds__(NG_SCAN_THREADS, 8) void chamfer_grid_kernel(
    int n, int m, int cells1, int cells2, int clouds, const float4* __restrict__ sorted1,
    const float4* __restrict__ sorted2, const float4* __restrict__ boxes1,
    const float4* __restrict__ boxes2, float* __restrict__ dist1, float* __restrict__ dist2,
    int32_t* __restrict__ idx1, int32_t* __restrict__ idx2, const int* __restrict__ wide1,
    const int* __restrict__ wide2, int window_cells, int part_cells, int log2_parts)
{
    __shared__ float4 stages[NG_SCAN_THREADS / TPK_WAVE][NG_CELL];
    extern __shared__ float lows_all[]; // [wavefronts][largest number of candidate cells, in whole groups of 64]

    const int lane = threadIdx.x & (TPK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TPK_WAVE);
    const int per_cloud = cells1 + cells2;
    const int64_t number = static_cast<int64_t>(xcd_local_block(blockIdx.x, gridDim.x)) *
                               (NG_SCAN_THREADS / TPK_WAVE) + wave;
    const int64_t task = number >> log2_parts;
    const int part = static_cast<int>(number) & ((1 << log2_parts) - 1);
    if (task >= static_cast<int64_t>(per_cloud) * clouds)
        return; // (no workgroup barrier anywhere in this kernel)
    int cloud = static_cast<int>(task / per_cloud);
    int r = static_cast<int>(task - static_cast<int64_t>(cloud) * per_cloud);
    if (window_cells > 0)
    {
        // Wavefronts start in the order of their numbers, and the call lasts as long as the wavefront that ends
        // last: the cells with the widest boxes - whose queries search longest - go first.  The cells of both
        // clouds' windows are dealt out in groups of NG_DEAL windows, window after window, every window
        // handing out its cells in the order the ordering kernel left: every part's wide ones first, then the others.
        const int per_cloud_windows = per_cloud / window_cells;
        const int64_t all_windows = static_cast<int64_t>(per_cloud_windows) * clouds;
        const int64_t group = task / (NG_DEAL * window_cells);
        const int within = static_cast<int>(task - group * (NG_DEAL * window_cells));
        const int dealt = static_cast<int>(tpk_min64(NG_DEAL, all_windows - group * NG_DEAL));
        const int64_t window = group * NG_DEAL + within % dealt;
        const int rank = within / dealt;
        cloud = static_cast<int>(window / per_cloud_windows);
        const int k = static_cast<int>(window - static_cast<int64_t>(cloud) * per_cloud_windows);
        const int windows1 = cells1 / window_cells;
        const bool in_second = k >= windows1;
        const int own = in_second ? k - windows1 : k; // the window's number in its cloud
        const int64_t at = in_second ? static_cast<int64_t>(cloud) * (per_cloud_windows - windows1) + own : static_cast<int64_t>(cloud) * windows1 + own;
        const int* __restrict__ order = (in_second ? wide2 : wide1) + at * window_cells;
        int wide_of[CURVE_PARTS]; // (parts that there are not: no cells)
#pragma unroll
        for (int p = 0; p < CURVE_PARTS; ++p)
            wide_of[p] = p * part_cells < window_cells ? order[p * part_cells] >> 16 : 0;
        int place = 0, left = rank; // the cell's place in `order`
        bool found = false;
#pragma unroll
        for (int turn = 0; turn < 2; ++turn)
#pragma unroll
            for (int p = 0; p < CURVE_PARTS; ++p)
            {
                const int size = max(min(part_cells, window_cells - p * part_cells), 0);
                const int count = turn == 0 ? wide_of[p] : size - wide_of[p];
                if (!found && left < count)
                {
                    place = p * part_cells + (turn == 0 ? left : wide_of[p] + left);
                    found = true;
                }
                left -= count;
            }
        r = (in_second ? cells1 : 0) + own * window_cells + (order[place] & 0xFFFF);
    }
    const bool second = r >= cells1;
    const int qcell = second ? r - cells1 : r;
    const int qcells = second ? cells2 : cells1;
    const int ccells = second ? cells1 : cells2;
    const int qcount = second ? m : n;
    const float4* __restrict__ qpts = (second ? sorted2 : sorted1) + static_cast<int64_t>(cloud) * qcells * NG_CELL;
    const float4* __restrict__ qbox = (second ? boxes2 : boxes1) + static_cast<int64_t>(cloud) * qcells * NG_BOX;
    const float4* __restrict__ cpts = (second ? sorted1 : sorted2) + static_cast<int64_t>(cloud) * ccells * NG_CELL;
    const float4* __restrict__ cbox = (second ? boxes1 : boxes2) + static_cast<int64_t>(cloud) * ccells * NG_BOX;
    const float4* __restrict__ cruns = (second ? boxes1 : boxes2) + static_cast<int64_t>(clouds) * ccells * NG_BOX +
                                       static_cast<int64_t>(cloud) * ccells * NG_RUN_BOXES;
    float* __restrict__ dout = (second ? dist2 : dist1) + static_cast<int64_t>(cloud) * qcount;
    int32_t* __restrict__ iout = (second ? idx2 : idx1) + static_cast<int64_t>(cloud) * qcount;
    float4* const stage = stages[wave];
    float* const lows = lows_all + wave * ((max(cells1, cells2) + NG_CELL - 1) / NG_CELL * NG_CELL);
    TPK_WORK_DECL
    TPK_PRODUCTS_DECL

    const float4 query = qpts[qcell * NG_CELL + lane];
    const float qx = query.x, qy = query.y, qz = query.z;
    // 0x7FFFFFFF: padding, nothing to store; so are the queries of the cell's other parts here
    const int qindex = ((lane << log2_parts) / TPK_WAVE) == part ? __float_as_int(query.w) : 0x7FFFFFFF;
    if (__ballot(qindex != 0x7FFFFFFF) == 0)
        return; // a cell without points (the last window of a cloud may have some)
    float4 qlo = qbox[qcell * NG_BOX + 0], qhi = qbox[qcell * NG_BOX + 1];
    if (log2_parts > 0)
        query_box(qx, qy, qz, qindex != 0x7FFFFFFF, qlo, qhi);

    const int groups = (ccells + NG_CELL - 1) / NG_CELL;
    const bool real = qindex != 0x7FFFFFFF;
    float best = __builtin_inff();
    int bi = 0x7FFFFFFF;
    // Box distances to all candidate cells, kept in the wavefront's LDS row (lane l computes
    // cells l, 64 + l, ...); +inf marks a cell that does not exist or has been scanned.
    unsigned seed_key = 0xFFFFFFFFu;
#pragma unroll 4 // (the boxes of four groups on their way at a time)
    for (int g = 0; g < groups; ++g)
    {
        const int c = g * NG_CELL + lane;
        const bool valid = c < ccells;
        const int cc = valid ? c : 0;
        const float4 clo = cbox[cc * NG_BOX + 0], chi = cbox[cc * NG_BOX + 1];
        const float lb = box_box_dist2(qlo, qhi, clo, chi);
        lows[c] = valid ? lb : __builtin_inff();
        // The first cell to scan: the one whose box centre is nearest to the centre of the queries'
        // box (many boxes overlap it; a good first answer lets the lanes turn most of them down).
        // The six lowest bits of the distance carry g.
        const float ex = (clo.x + chi.x) - (qlo.x + qhi.x), ey = (clo.y + chi.y) - (qlo.y + qhi.y);
        const float ez = (clo.z + chi.z) - (qlo.z + qhi.z);
        const float centre = __builtin_fmaf(ex, ex, __builtin_fmaf(ey, ey, ez * ez));
        const unsigned key = (static_cast<unsigned>(__float_as_int(centre)) & ~63u) | static_cast<unsigned>(g);
        seed_key = valid && lb < __builtin_inff() && key < seed_key ? key : seed_key;
    }
    const unsigned lowest = wave_min_u32(seed_key);
    int seed = static_cast<int>(lowest & 63u) * NG_CELL + __builtin_ctzll(__ballot(seed_key == lowest));
    if (seed >= ccells) // no lane had a usable key (NaN boxes)
        seed = 0;

    // The units of the matrix scan: 512 to 1024 for the largest distance, along one axis, from the centre of the queries' box
    // to their own and the first cell's faces (a query's answer is at most twice that away from its query).  Where the
    // first cell is far away for its size and that of the queries' box, all its points are about equally distant and
    // the products could not tell them apart.
    MatrixFrame frame;
    bool matrix;
    {
        const float4 slo = cbox[seed * NG_BOX + 0], shi = cbox[seed * NG_BOX + 1];
        const float cx = 0.5f * (qlo.x + qhi.x), cy = 0.5f * (qlo.y + qhi.y), cz = 0.5f * (qlo.z + qhi.z);
        const float own = fmaxf(fmaxf(qhi.x - cx, qhi.y - cy), qhi.z - cz);
        const float extent = fmaxf(own, 0.5f * fmaxf(fmaxf(shi.x - slo.x, shi.y - slo.y), shi.z - slo.z));
        const float radius = fmaxf(fmaxf(fmaxf(fabsf(slo.x - cx), fabsf(shi.x - cx)), fmaxf(fabsf(slo.y - cy), fabsf(shi.y - cy))),
                                   fmaxf(fmaxf(fabsf(slo.z - cz), fabsf(shi.z - cz)), own));
        const int exponent = (__float_as_int(radius) >> 23) - 127;
        frame.scale = __int_as_float((127 + 9 - exponent) << 23);
        frame.ox = -cx * frame.scale;
        frame.oy = -cy * frame.scale;
        frame.oz = -cz * frame.scale;
        frame.minus_one = to_vector_register(-1.f);
        matrix = radius >= 8.9e-16f && radius <= 1.1e15f && radius <= MX_NEAR * extent; // (false for what is not a number)
    }
    float x = __builtin_fmaf(qx, frame.scale, frame.ox), y = __builtin_fmaf(qy, frame.scale, frame.oy), z = __builtin_fmaf(qz, frame.scale, frame.oz);
    matrix = matrix && __ballot(real && !(fabsf(x) <= 1100.f && fabsf(y) <= 1100.f && fabsf(z) <= 1100.f)) == 0;
    Nearest s;
    s.best = real ? __builtin_inff() : -1.f; // (a padding lane never asks for a scan)
    s.chunk = 0;
    s.tie = false;
    bool ask = real; // left to the exact scan
    bool tie = false; // left to the pass behind it
    float reach = __builtin_inff();
    int scans = 0; // behind the first cell's
    if (matrix)
    {
        x = real ? x : 0.f;
        y = real ? y : 0.f;
        z = real ? z : 0.f;
        const float square = __builtin_fmaf(x, x, __builtin_fmaf(y, y, z * z));
        const float own_error = __builtin_fmaf(square, MX_ERROR, 0.0625f);
        const float unit = 1.f / (frame.scale * frame.scale);
        const float reach_factor = (1.f + MX_ERROR_NEAR) * unit, reach_error = own_error * unit;
        half8_t queries[2];
        {
            half2_t xy_high, xy_low, z_high, z_low, s_high, s_low;
            split_half(-2.f * x, -2.f * y, frame.minus_one, xy_high, xy_low);
            split_half(-2.f * z, 0.f, frame.minus_one, z_high, z_low);
            split_half(square * (1.f / MX_FAR), 0.f, frame.minus_one, s_high, s_low);
            const half2_t zs = half2_t{z_high[0], static_cast<_Float16>(MX_FAR)};
            tile_operands({xy_high, xy_high, zs, zs}, {xy_low, xy_low, half2_t{z_low[0], 0}, half2_t{s_high[0], s_low[0]}}, queries);
        }
        MatrixNearest near[2];
        near[0].m1 = near[0].m2 = near[1].m1 = near[1].m2 = __float_as_int(__builtin_inff());
        near[0].cell = near[1].cell = seed;
        matrix_scan(cpts, seed, __ballot(real), lane, frame, queries, near TPK_PRODUCTS_ARG);
        // The smallest product of the lane's query, and the squared distance that holds the query's answer for certain.  (A tile
        // without a query is never scanned: its m1 stay infinite.  No lane without a query may reach for anything.)
        auto smallest = [&]() {
            int a, b;
            by_query(near[0].m1, near[1].m1, a, b);
            return __int_as_float(max(min(a, b), 0));
        };
        float m = smallest();
        auto reach_of = [&](float product) { return real ? __builtin_fmaf(product, reach_factor, reach_error) : -1.f; };
        reach = reach_of(m);
        // The second smallest, and whether the smallest is surely further from it than both err.
        auto second_smallest = [&]() {
            int a, b, a2, b2;
            by_query(near[0].m1, near[1].m1, a, b);
            by_query(near[0].m2, near[1].m2, a2, b2);
            return __int_as_float(min(min(a2, b2), max(a, b)));
        };
        auto clear = [&](float second) { return second > m + 2.f * __builtin_fmaf(m, MX_ERROR_NEAR, own_error) && m < MX_LIMIT; };
        // Where the first cell's second smallest products are near the error already, or near the smallest, the search would leave the queries
        // over.  (A wavefront that shares its cell has half of the queries at most and keeps to the first test: it would give few back.)
        float m2 = second_smallest();
        const bool alone = log2_parts == 0;
        const int close = __builtin_popcountll(__ballot(real && (m2 < MX_CLOSE * own_error || (alone && !clear(m2)))));
        if (close <= (alone ? MX_MANY : 2 * MX_MANY))
        {
            // First the cells whose boxes overlap the queries' box - they hold nearly all the answers - then whatever
            // the worst answer still admits (a cell is looked at once: answers only get better).
            bool given_up = false;
            for (int phase = 0; phase < 2; ++phase)
            {
                if (phase == 1)
                {
                    m = smallest();
                    m2 = second_smallest();
                    const unsigned long long unclear = __ballot(real && !clear(m2)), blind = unclear & __ballot(m < own_error);
                    const int count = __builtin_popcountll(unclear);
                    given_up = count > MX_MOST && count * MX_SCANS > scans && 2 * __builtin_popcountll(blind) <= count;
                    if (given_up)
                        break;
                }
                for (int g = 0; g < groups; ++g)
                {
                    const float lw = lows[g * NG_CELL + lane];
                    float bound = __int_as_float(wave_max_i32(__float_as_int(reach)));
                    unsigned long long live =
                        __ballot(phase == 0 ? lw == 0.f : lw > 0.f && lw < __builtin_inff() && lw * NG_MARGIN <= bound);
                    if (g == seed / NG_CELL)
                        live &= ~(1ull << (seed % NG_CELL));
                    while (live != 0)
                    {
                        const int c = g * NG_CELL + __builtin_ctzll(live);
                        live &= live - 1;
                        const float lb = point_box_dist2(qx, qy, qz, cbox[c * NG_BOX + 0], cbox[c * NG_BOX + 1]);
                        const unsigned long long want = __ballot(lb * NG_MARGIN <= reach);
                        if (want == 0)
                            continue;
                        matrix_scan(cpts, c, want, lane, frame, queries, near TPK_PRODUCTS_ARG);
                        reach = reach_of(smallest());
                        ++scans;
                        if (phase)
                        {
                            bound = __int_as_float(wave_max_i32(__float_as_int(reach)));
                            live &= __ballot(lw * NG_MARGIN <= bound);
                        }
                    }
                }
            }
            m = smallest();
            m2 = second_smallest();
            ask = real && (given_up || !clear(m2));
        }
        // The eight of the smallest product: the answer of a query that is not left over, and no further away than it for one that is.
        int a, b, cell_a, cell_b;
        by_query(near[0].m1, near[1].m1, a, b);
        by_query(near[0].cell, near[1].cell, cell_a, cell_b);
        const int first = (a <= b ? cell_a : cell_b) * NG_CELL + (min(a, b) & 3) * 16 + (a <= b ? 0 : 4);
#pragma unroll
        for (int c = 0; c < 8; ++c) // (rows 0 .. 3 and 8 .. 11 of 16, or those four further on)
        {
            const float4 p = cpts[first + (c & 3) + 2 * (c & 4)];
            const float d = tpk_dist2(p.x, p.y, p.z, qx, qy, qz);
            const int ci = __float_as_int(p.w);
            bi = d < best || (d == best && ci < bi) ? ci : bi;
            best = fminf(d, best);
        }
        TPK_WORK_ADD(8);
        // The answer of a query that is left over is below its reach, not equal, and no more than the best of the eight.
        reach = m < MX_LIMIT ? reach : __builtin_inff();
        reach = fminf(reach, __int_as_float(min(__float_as_int(best), 0x7F7FFFFF) + 1));
        const int left = __builtin_popcountll(__ballot(ask)), blind = __builtin_popcountll(__ballot(ask && m < own_error));
        if (left <= MX_PASS || (left * MX_SCANS <= scans && 2 * blind <= left))
        {
            tie = ask;
            ask = false;
        }
        s.best = ask ? reach : -1.f;
    }
    if (__ballot(ask) != 0)
    {
        if (!matrix)
        {
            scan_cell(cpts, cruns, seed, stage, lane, qx, qy, qz, s TPK_WORK_ARG);
            if (lane == (seed & (NG_CELL - 1)))
                lows[seed] = __builtin_inff();
        }
        // (in the same order)
        for (int phase = 0; phase < 2; ++phase)
            for (int g = 0; g < groups; ++g)
            {
                const float lw = lows[g * NG_CELL + lane];
                float bound = __int_as_float(wave_max_i32(__float_as_int(s.best)));
                unsigned long long live =
                    __ballot(lw < __builtin_inff() && (phase == 0 ? lw == 0.f : lw * NG_MARGIN <= bound));
                while (live != 0)
                {
                    const int bit = __builtin_ctzll(live);
                    const int c = g * NG_CELL + bit;
                    live &= live - 1;
                    const float lb = point_box_dist2(qx, qy, qz, cbox[c * NG_BOX + 0], cbox[c * NG_BOX + 1]);
                    const unsigned long long want = __ballot(lb * NG_MARGIN <= s.best);
                    // scanned, or no lane can improve here now - and answers only get better: never again
                    if (lane == bit)
                        lows[c] = __builtin_inff();
                    if (want == 0)
                        continue;
                    if (__builtin_popcountll(want) <= NG_FEW)
                        scan_cell_few(cpts, c, want, lane, qx, qy, qz, s TPK_WORK_ARG);
                    else
                        scan_cell(cpts, cruns, c, stage, lane, qx, qy, qz, s TPK_WORK_ARG);
                    if (phase)
                    {
                        bound = __int_as_float(wave_max_i32(__float_as_int(s.best)));
                        live &= __ballot(lw * NG_MARGIN <= bound);
                    }
                }
            }

        // The index: lowest original index among the candidates of the recorded group that are at
        // the minimum distance (re-evaluated with the same operations, hence the same bits).
        best = ask ? s.best : best;
        bi = ask ? 0x7FFFFFFF : bi;
#pragma unroll
        for (int c = 0; c < NG_CHUNK; ++c)
        {
            const float4 p = cpts[s.chunk * NG_CHUNK + c];
            const float d = tpk_dist2(p.x, p.y, p.z, qx, qy, qz);
            const int ci = __float_as_int(p.w);
            bi = (ask && d == best && ci < bi) ? ci : bi;
        }
        TPK_WORK_ADD(NG_CHUNK);
        reach = ask ? best : reach;
        tie = tie || (ask && s.tie);
    }
    // Several groups reached a query's minimum (about one query in 10^5 on random clouds, every query on a lattice), or
    // came too close to it for the products to tell (one in 1200 to 5500): the nearest candidate, of several the one of lowest index,
    // over all cells within reach.  One such query at a time: the lanes test the boxes of all cells side by side, then the
    // candidates of every cell that passes.
    for (unsigned long long tied = __ballot(tie); tied != 0; tied &= tied - 1)
    {
        const int q = __builtin_ctzll(tied);
        const float ux = tpk_read_lane(qx, q), uy = tpk_read_lane(qy, q), uz = tpk_read_lane(qz, q);
        const float ub = tpk_read_lane(reach, q);
        float nearest = __builtin_inff();
        int lowest = 0x7FFFFFFF;
        auto look = [&](auto batch, int g0) __attribute__((always_inline)) {
            constexpr int BATCH = batch.value; // groups whose boxes are on their way at a time
            unsigned long long cells[BATCH];
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
            {
                const int c = (g0 + u) * NG_CELL + lane;
                const int cc = c < ccells ? c : 0;
                const float lb = point_box_dist2(ux, uy, uz, cbox[cc * NG_BOX + 0], cbox[cc * NG_BOX + 1]);
                cells[u] = __ballot(c < ccells && lb * NG_MARGIN <= ub);
            }
#pragma unroll
            for (int v = 0; v < BATCH; ++v)
                while (cells[v] != 0)
                {
                    TPK_WORK_ADD(min(4, __builtin_popcountll(cells[v])));
                    float4 p[4]; // (four cells on their way at a time; behind the last, the last one again)
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                    {
                        p[u] = cpts[((g0 + v) * NG_CELL + __builtin_ctzll(cells[v])) * NG_CELL + lane];
                        const unsigned long long rest = cells[v] & (cells[v] - 1);
                        cells[v] = rest != 0 || u == 3 ? rest : cells[v];
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                    {
                        const float d = tpk_dist2(p[u].x, p[u].y, p[u].z, ux, uy, uz);
                        const int ci = __float_as_int(p[u].w);
                        lowest = d < nearest || (d == nearest && ci < lowest) ? ci : lowest;
                        nearest = d < nearest ? d : nearest;
                    }
                }
        };
        int g0 = 0;
        for (; g0 + 4 <= groups; g0 += 4)
            look(std::integral_constant<int, 4>{}, g0);
        for (; g0 < groups; ++g0)
            look(std::integral_constant<int, 1>{}, g0);
        // (distances are >= +0: their bit patterns order like integers)
        const float least = __int_as_float(wave_min_i32(__float_as_int(nearest)));
        lowest = wave_min_i32(nearest == least ? lowest : 0x7FFFFFFF);
        best = lane == q ? least : best;
        bi = lane == q ? lowest : bi;
    }
    TPK_WORK_FLUSH
    TPK_PRODUCTS_FLUSH
    if (real)
    {
        dout[qindex] = best;
        iout[qindex] = bi == 0x7FFFFFFF ? 0 : bi;
    }
}

// ---------------------------------------------------------------------------------------
// three_nn over cells: the three nearest known points of every unknown point.
//
// The running answer of a lane is a triple sorted by (distance, original index); a candidate
// enters where it is smaller in that order.  This is the order a serial scan in index order with
// strictly-smaller replacement (cuda/src/interpolate_gpu.cu:9-65) ends with, whatever order the
// candidates are visited in.  A cell is skipped when its box is further away than the third
// best of every lane.
// ---------------------------------------------------------------------------------------
struct Nearest3
{
    float b1, b2, b3;
    int i1, i2, i3;
};

__device__ __forceinline__ bool pair_less(float d, int ci, float b, int i)
{
    return d < b || (d == b && ci < i);
}

__device__ __forceinline__ void scan_cell3(const float4* __restrict__ cand, const float4* __restrict__ runs,
                                           int cell, float4* stage, int lane, float qx, float qy, float qz,
                                           Nearest3& s TPK_WORK_PARAM)
{
    stage[lane] = cand[cell * NG_CELL + lane];
    // (the boxes of the cell's four runs are requested together with its candidates: one wait, not five)
    float4 quarter[NG_RUN_BOXES];
#pragma unroll
    for (int i = 0; i < NG_RUN_BOXES; ++i)
        quarter[i] = runs[cell * NG_RUN_BOXES + i];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    bool reached = true;
#pragma unroll
    for (int ch = 0; ch < NG_CELL / NG_CHUNK; ++ch)
    {
        // a run of 16 candidates whose box no lane's third best reaches is passed over
        // (decided at the run's first group: `reached` carries it to the second)
        if ((ch & 1) == 0)
        {
            const float lb = point_box_dist2(qx, qy, qz, quarter[ch], quarter[ch + 1]);
            reached = __ballot(lb * NG_MARGIN <= s.b3) != 0;
        }
        if (!reached)
            continue;
        float mn = 0.f;
        float ds[NG_CHUNK];
        int cis[NG_CHUNK];
#pragma unroll
        for (int c = 0; c < NG_CHUNK; ++c)
        {
            const float4 p = stage[ch * NG_CHUNK + c];
            // Operand order of the reference: (query - scanned).
            ds[c] = tpk_dist2(qx, qy, qz, p.x, p.y, p.z);
            cis[c] = __float_as_int(p.w);
            mn = c == 0 ? ds[c] : fminf(mn, ds[c]);
        }
        TPK_WORK_ADD(NG_CHUNK);
        if (__ballot(mn <= s.b3) == 0)
            continue; // no candidate of this group enters any lane's triple
#pragma unroll
        for (int c = 0; c < NG_CHUNK; ++c)
        {
            const float d = ds[c];
            const int ci = cis[c];
            const bool l3 = pair_less(d, ci, s.b3, s.i3);
            if (__ballot(l3) == 0)
                continue;
            const bool l2 = pair_less(d, ci, s.b2, s.i2);
            const bool l1 = pair_less(d, ci, s.b1, s.i1);
            s.b3 = l2 ? s.b2 : (l3 ? d : s.b3);
            s.i3 = l2 ? s.i2 : (l3 ? ci : s.i3);
            s.b2 = l1 ? s.b1 : (l2 ? d : s.b2);
            s.i2 = l1 ? s.i1 : (l2 ? ci : s.i2);
            s.b1 = l1 ? d : s.b1;
            s.i1 = l1 ? ci : s.i1;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One wavefront = the 64 unknown points of one cell; logical wavefront = cloud * qcells + cell.
// The same for a cell that only a few queries of the wavefront still ask for: one query at a time, the
// 64 candidates of the cell side by side in the lanes (`want`: the lanes whose queries ask).  The candidates
// that enter the query's triple are taken smallest first in the triple's order (distance, then index); no
// more than three of them can stay.
constexpr int NG_FEW3 = 8; // (uniform clouds, 16 x 16384 queries: 0 / 4 / 8 / 12 / 16: 98.7 / 95.1 / 94.9 / 95.6 / 99.8 us)
__device__ __forceinline__ void scan_cell3_few(const float4* __restrict__ cand, int cell, unsigned long long want,
                                               int lane, float qx, float qy, float qz, Nearest3& s TPK_WORK_PARAM)
{
    const float4 p = cand[cell * NG_CELL + lane];
    const int ci = __float_as_int(p.w);
    while (want != 0)
    {
        const int q = __builtin_ctzll(want);
        want &= want - 1;
        TPK_WORK_ADD(1);
        const float ux = tpk_read_lane(qx, q), uy = tpk_read_lane(qy, q), uz = tpk_read_lane(qz, q);
        // Operand order of the reference: (query - scanned).
        const float d = tpk_dist2(ux, uy, uz, p.x, p.y, p.z);
        unsigned long long in = __ballot(pair_less(d, ci, tpk_read_lane(s.b3, q), tpk_read_lane(s.i3, q)));
        for (int r = 0; r < 3 && in != 0; ++r)
        {
            // distances are >= +0: their bit patterns order like integers
            const bool mine = (in >> lane) & 1ull;
            const int least = wave_min_i32(mine ? __float_as_int(d) : 0x7FFFFFFF);
            unsigned long long at = __ballot(mine && __float_as_int(d) == least);
            if (at & (at - 1)) // equal distances: the lowest index
            {
                const bool tied = (at >> lane) & 1ull;
                const int first = wave_min_i32(tied ? ci : 0x7FFFFFFF);
                at = __ballot(tied && ci == first);
            }
            const int from = __builtin_ctzll(at);
            in &= ~(1ull << from);
            const float dv = __int_as_float(least);
            const int cv = tpk_read_lane(ci, from);
            if (lane == q)
            {
                const bool l3 = pair_less(dv, cv, s.b3, s.i3);
                const bool l2 = pair_less(dv, cv, s.b2, s.i2);
                const bool l1 = pair_less(dv, cv, s.b1, s.i1);
                s.b3 = l2 ? s.b2 : (l3 ? dv : s.b3);
                s.i3 = l2 ? s.i2 : (l3 ? cv : s.i3);
                s.b2 = l1 ? s.b1 : (l2 ? dv : s.b2);
                s.i2 = l1 ? s.i1 : (l2 ? cv : s.i2);
                s.b1 = l1 ? dv : s.b1;
                s.i1 = l1 ? cv : s.i1;
            }
        }
    }
}

// Where the queries' cells are too few to fill the chip, the search lasts as long as its slowest wavefront, one whose 64 queries lie far
// apart and ask for many cells, one after the other.  The queries of a cell are then shared by 2, 4 or 8 wavefronts, whose boxes
// are smaller and which scan fewer cells each, as long as these are no more than four per SIMD: beyond, the scans that
// several of them repeat cost more than the tail (16 x 16384 queries on as many points 110 us whole, in halves 119; on 4096, eight
// clusters, 120 and 124).  us, whole -> as here, even / eight clusters / sphere: 1 x 16384 on as many 91 -> 54 / 256 -> 114 / 89 -> 52; 2 x 16384 91 -> 60 /
// 256 -> 112 / 94 -> 59; 4 x 16384 91 -> 66 / 255 -> 167 / 93 -> 67; 8 x 16384 91 -> 80 / 256 -> 215 / 96 -> 90; 2 x 60000 216 -> 157 / 548 -> 458 /
// 184 -> 157; clusters handed over by the grid in LDS, 1 x 4096 106 -> 63, 8 x 4096 128 -> 101, 4 x 8264 on 4132 106 -> 97, 16 x 2000 85 -> 79.
constexpr int64_t NG_PARTED_WAVES = 4096;
constexpr int NG_MOST_PARTS = 3; // log2: 8 queries per wavefront
__global__ __launch_bounds__(NG_SCAN_THREADS) void three_nn_grid_kernel(
    int n, int m, int qcells, int ccells, int clouds, const float4* __restrict__ sorted_unknown,
    const float4* __restrict__ sorted_known, const float4* __restrict__ boxes_known, float* __restrict__ dist2,
    int32_t* __restrict__ idx, bool root, const int* __restrict__ only, int log2_parts)
{
    __shared__ float4 stages[NG_SCAN_THREADS / TPK_WAVE][NG_CELL];
    extern __shared__ float lows_all[]; // [wavefronts][candidate cells, in whole groups of 64]

    const int lane = threadIdx.x & (TPK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TPK_WAVE);
    const int64_t task = static_cast<int64_t>(xcd_local_block(blockIdx.x, gridDim.x)) *
                             (NG_SCAN_THREADS / TPK_WAVE) + wave;
    const int64_t cell_task = task >> log2_parts;
    if (cell_task >= static_cast<int64_t>(qcells) * clouds)
        return; // (no workgroup barrier anywhere in this kernel)
    const int cloud = static_cast<int>(cell_task / qcells);
    if (only && only[cloud] == 0)
        return; // (a cloud that another kernel has answered)
    const int qcell = static_cast<int>(cell_task - static_cast<int64_t>(cloud) * qcells);
    const int part = static_cast<int>(task) & ((1 << log2_parts) - 1);
    const float4* __restrict__ qpts = sorted_unknown + static_cast<int64_t>(cloud) * qcells * NG_CELL;
    const float4* __restrict__ cpts = sorted_known + static_cast<int64_t>(cloud) * ccells * NG_CELL;
    const float4* __restrict__ cbox = boxes_known + static_cast<int64_t>(cloud) * ccells * NG_BOX;
    const float4* __restrict__ cruns =
        boxes_known + static_cast<int64_t>(clouds) * ccells * NG_BOX + static_cast<int64_t>(cloud) * ccells * NG_RUN_BOXES;
    dist2 += static_cast<int64_t>(cloud) * n * 3;
    idx += static_cast<int64_t>(cloud) * n * 3;
    float4* const stage = stages[wave];
    float* const lows = lows_all + wave * ((ccells + NG_CELL - 1) / NG_CELL * NG_CELL);
    TPK_WORK_DECL

    const float4 query = qpts[qcell * NG_CELL + lane];
    const float qx = query.x, qy = query.y, qz = query.z;
    // 0x7FFFFFFF: padding, nothing to store; so are the queries of the cell's other parts here
    const int qindex = ((lane << log2_parts) / TPK_WAVE) == part ? __float_as_int(query.w) : 0x7FFFFFFF;
    if (__ballot(qindex != 0x7FFFFFFF) == 0)
        return; // a cell without points (the last window of a cloud may have some)
    float4 qlo, qhi;
    query_box(qx, qy, qz, qindex != 0x7FFFFFFF, qlo, qhi);

    const int groups = (ccells + NG_CELL - 1) / NG_CELL;
    unsigned seed_key = 0xFFFFFFFFu;
#pragma unroll 4 // (the boxes of four groups on their way at a time: clusters 2 x 60000 551 -> 533 us, 16 x 16384 263 -> 258)
    for (int g = 0; g < groups; ++g)
    {
        const int c = g * NG_CELL + lane;
        const bool valid = c < ccells;
        const int cc = valid ? c : 0;
        const float4 clo = cbox[cc * NG_BOX + 0], chi = cbox[cc * NG_BOX + 1];
        const float lb = box_box_dist2(qlo, qhi, clo, chi);
        lows[c] = valid ? lb : __builtin_inff();
        // the first cell to scan: nearest box centre (the six lowest bits of the distance carry g)
        const float ex = (clo.x + chi.x) - (qlo.x + qhi.x), ey = (clo.y + chi.y) - (qlo.y + qhi.y);
        const float ez = (clo.z + chi.z) - (qlo.z + qhi.z);
        const float centre = __builtin_fmaf(ex, ex, __builtin_fmaf(ey, ey, ez * ez));
        const unsigned key = (static_cast<unsigned>(__float_as_int(centre)) & ~63u) | static_cast<unsigned>(g);
        seed_key = valid && lb < __builtin_inff() && key < seed_key ? key : seed_key;
    }
    Nearest3 s;
    s.b1 = s.b2 = s.b3 = qindex == 0x7FFFFFFF ? -1.f : __builtin_inff(); // (a padding lane never asks for a scan)
    s.i1 = s.i2 = s.i3 = 0;
    {
        const unsigned lowest = wave_min_u32(seed_key);
        int seed = static_cast<int>(lowest & 63u) * NG_CELL + __builtin_ctzll(__ballot(seed_key == lowest));
        if (seed >= ccells)
            seed = 0;
        scan_cell3(cpts, cruns, seed, stage, lane, qx, qy, qz, s TPK_WORK_ARG);
        if (lane == (seed & (NG_CELL - 1)))
            lows[seed] = __builtin_inff();
    }
    for (int phase = 0; phase < 2; ++phase)
        for (int g = 0; g < groups; ++g)
        {
            const float lw = lows[g * NG_CELL + lane];
            float bound = __int_as_float(wave_max_i32(__float_as_int(s.b3)));
            unsigned long long live =
                __ballot(lw < __builtin_inff() && (phase == 0 ? lw == 0.f : lw * NG_MARGIN <= bound));
            while (live != 0)
            {
                const int bit = __builtin_ctzll(live);
                const int c = g * NG_CELL + bit;
                live &= live - 1;
                const float lb = point_box_dist2(qx, qy, qz, cbox[c * NG_BOX + 0], cbox[c * NG_BOX + 1]);
                const unsigned long long want = __ballot(lb * NG_MARGIN <= s.b3);
                if (want != 0 && __builtin_popcountll(want) <= NG_FEW3)
                    scan_cell3_few(cpts, c, want, lane, qx, qy, qz, s TPK_WORK_ARG);
                else if (want != 0)
                    scan_cell3(cpts, cruns, c, stage, lane, qx, qy, qz, s TPK_WORK_ARG);
                if (lane == bit)
                    lows[c] = __builtin_inff(); // scanned, or useless now and ever after
                if (phase)
                {
                    bound = __int_as_float(wave_max_i32(__float_as_int(s.b3)));
                    live &= __ballot(lw * NG_MARGIN <= bound);
                }
            }
        }
    TPK_WORK_FLUSH
    if (qindex != 0x7FFFFFFF)
    {
        dist2[qindex * 3 + 0] = root ? sqrtf(s.b1) : s.b1;
        dist2[qindex * 3 + 1] = root ? sqrtf(s.b2) : s.b2;
        dist2[qindex * 3 + 2] = root ? sqrtf(s.b3) : s.b3;
        idx[qindex * 3 + 0] = s.i1;
        idx[qindex * 3 + 1] = s.i2;
        idx[qindex * 3 + 2] = s.i3;
    }
}

// ---------------------------------------------------------------------------------------
// k nearest neighbours over cells: three_nn's search with a list of up to 32 entries per lane
// (topk.h).  A larger k is served in rounds: round r finds the entries 32 r .. 32 r + 31, which
// are the smallest pairs after the last one of the round before.  A cell is skipped when its box
// is further away than the last kept entry of every lane.
// ---------------------------------------------------------------------------------------
template <int K>
__device__ __forceinline__ void scan_cell_k(const float4* __restrict__ cand, const float4* __restrict__ runs,
                                            int cell, float4* stage, int lane, float qx, float qy, float qz,
                                            NearestK<K>& s)
{
    stage[lane] = cand[cell * NG_CELL + lane];
    float worst = s.worst(); // distance of the lane's last entry
    // The runs of 16 candidates whose box no lane's last entry reaches are passed over.  The four boxes are
    // requested together with the candidates and tested before the scan: one wait, not five.
    unsigned reached = 0;
    {
        float4 quarter[NG_RUN_BOXES];
#pragma unroll
        for (int i = 0; i < NG_RUN_BOXES; ++i)
            quarter[i] = runs[cell * NG_RUN_BOXES + i];
#pragma unroll
        for (int run = 0; run < NG_RUN_BOXES / 2; ++run)
        {
            const float lb = point_box_dist2(qx, qy, qz, quarter[2 * run], quarter[2 * run + 1]);
            reached |= __ballot(lb * NG_MARGIN <= worst) != 0 ? 1u << run : 0u;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    for (int ch = 0; ch < NG_CELL / NG_CHUNK; ++ch)
    {
        if (((reached >> (ch >> 1)) & 1u) == 0)
            continue;
        float mn = 0.f;
        float ds[NG_CHUNK];
        int cis[NG_CHUNK];
#pragma unroll
        for (int c = 0; c < NG_CHUNK; ++c)
        {
            const float4 p = stage[ch * NG_CHUNK + c];
            ds[c] = tpk_dist2(qx, qy, qz, p.x, p.y, p.z);
            cis[c] = __float_as_int(p.w);
            mn = c == 0 ? ds[c] : fminf(mn, ds[c]);
        }
        if (__ballot(mn <= worst) == 0)
            continue; // no candidate of this group enters any lane's list
#pragma unroll
        for (int c = 0; c < NG_CHUNK; ++c)
        {
            const unsigned long long cand = knn_key(ds[c], cis[c]);
            const bool in = s.admits(cand);
            if (__ballot(in) == 0)
                continue;
            if (in)
                s.insert(cand);
        }
        worst = s.worst();
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One wavefront = the 64 queries of one cell; logical wavefront = cloud * qcells + cell.
// first: number of entries found by earlier rounds; count: entries this round finds (<= K).
template <int K>
__global__ __launch_bounds__(NG_SCAN_THREADS) void knn_grid_kernel(
    int n, int k, int first, int count, float limit, int qcells, int ccells, int clouds,
    const float4* __restrict__ sorted_query, const float4* __restrict__ sorted_support,
    const float4* __restrict__ boxes_support, float* __restrict__ dist2, int64_t* __restrict__ idx)
{
    __shared__ float4 stages[NG_SCAN_THREADS / TPK_WAVE][NG_CELL];
    extern __shared__ float lows_all[]; // [wavefronts][candidate cells, in whole groups of 64]

    const int lane = threadIdx.x & (TPK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TPK_WAVE);
    const int64_t task = static_cast<int64_t>(xcd_local_block(blockIdx.x, gridDim.x)) *
                             (NG_SCAN_THREADS / TPK_WAVE) + wave;
    if (task >= static_cast<int64_t>(qcells) * clouds)
        return; // (no workgroup barrier anywhere in this kernel)
    const int cloud = static_cast<int>(task / qcells);
    const int qcell = static_cast<int>(task - static_cast<int64_t>(cloud) * qcells);
    const float4* __restrict__ qpts = sorted_query + static_cast<int64_t>(cloud) * qcells * NG_CELL;
    const float4* __restrict__ cpts = sorted_support + static_cast<int64_t>(cloud) * ccells * NG_CELL;
    const float4* __restrict__ cbox = boxes_support + static_cast<int64_t>(cloud) * ccells * NG_BOX;
    const float4* __restrict__ cruns =
        boxes_support + static_cast<int64_t>(clouds) * ccells * NG_BOX + static_cast<int64_t>(cloud) * ccells * NG_RUN_BOXES;
    dist2 += static_cast<int64_t>(cloud) * n * k;
    idx += static_cast<int64_t>(cloud) * n * k;
    float4* const stage = stages[wave];
    float* const lows = lows_all + wave * ((ccells + NG_CELL - 1) / NG_CELL * NG_CELL);

    const float4 query = qpts[qcell * NG_CELL + lane];
    const float qx = query.x, qy = query.y, qz = query.z;
    const int qindex = __float_as_int(query.w); // 0x7FFFFFFF: padding, nothing to store
    if (__ballot(qindex != 0x7FFFFFFF) == 0)
        return; // a cell without points (the last window of a cloud may have some)
    const bool real = qindex != 0x7FFFFFFF;
    float4 qlo, qhi;
    query_box(qx, qy, qz, real, qlo, qhi);

    NearestK<K> s;
    {
        // the last pair of the round before (rounds of one call run one after the other)
        const int64_t at = static_cast<int64_t>(real ? qindex : 0) * k + first - 1;
        const bool later = first > 0 && real;
        s.reset(first > 0, later ? dist2[at] : 0.f, later ? static_cast<int>(idx[at]) : 0, !real, limit);
    }

    const int groups = (ccells + NG_CELL - 1) / NG_CELL;
    unsigned seed_key = 0xFFFFFFFFu;
    for (int g = 0; g < groups; ++g)
    {
        const int c = g * NG_CELL + lane;
        const bool valid = c < ccells;
        const int cc = valid ? c : 0;
        const float4 clo = cbox[cc * NG_BOX + 0], chi = cbox[cc * NG_BOX + 1];
        const float lb = box_box_dist2(qlo, qhi, clo, chi);
        lows[c] = valid ? lb : __builtin_inff();
        // the first cell to scan: nearest box centre (the six lowest bits of the distance carry g)
        const float ex = (clo.x + chi.x) - (qlo.x + qhi.x), ey = (clo.y + chi.y) - (qlo.y + qhi.y);
        const float ez = (clo.z + chi.z) - (qlo.z + qhi.z);
        const float centre = __builtin_fmaf(ex, ex, __builtin_fmaf(ey, ey, ez * ez));
        const unsigned key = (static_cast<unsigned>(__float_as_int(centre)) & ~63u) | static_cast<unsigned>(g);
        seed_key = valid && lb < __builtin_inff() && key < seed_key ? key : seed_key;
    }
    {
        const unsigned lowest = wave_min_u32(seed_key);
        int seed = static_cast<int>(lowest & 63u) * NG_CELL + __builtin_ctzll(__ballot(seed_key == lowest));
        if (seed >= ccells)
            seed = 0;
        scan_cell_k<K>(cpts, cruns, seed, stage, lane, qx, qy, qz, s);
        if (lane == (seed & (NG_CELL - 1)))
            lows[seed] = __builtin_inff();
    }
    for (int phase = 0; phase < 2; ++phase)
        for (int g = 0; g < groups; ++g)
        {
            const float lw = lows[g * NG_CELL + lane];
            float bound = __int_as_float(wave_max_i32(__float_as_int(s.worst())));
            unsigned long long live =
                __ballot(lw < __builtin_inff() && (phase == 0 ? lw == 0.f : lw * NG_MARGIN <= bound));
            while (live != 0)
            {
                const int bit = __builtin_ctzll(live);
                const int c = g * NG_CELL + bit;
                live &= live - 1;
                const float lb = point_box_dist2(qx, qy, qz, cbox[c * NG_BOX + 0], cbox[c * NG_BOX + 1]);
                if (__ballot(lb * NG_MARGIN <= s.worst()) != 0)
                    scan_cell_k<K>(cpts, cruns, c, stage, lane, qx, qy, qz, s);
                if (lane == bit)
                    lows[c] = __builtin_inff(); // scanned, or useless now and ever after
                if (phase)
                {
                    bound = __int_as_float(wave_max_i32(__float_as_int(s.worst())));
                    live &= __ballot(lw * NG_MARGIN <= bound);
                }
            }
        }
    if (real)
    {
#pragma unroll
        for (int j = 0; j < K; ++j)
            if (j < count)
            {
                dist2[static_cast<int64_t>(qindex) * k + first + j] = s.dist(j);
                idx[static_cast<int64_t>(qindex) * k + first + j] = s.index(j);
            }
    }
}

constexpr int NG_RUN = 16; // consecutive cells that share a second-level box in the wavefront-per-query search

// ---------------------------------------------------------------------------------------
// Ball query over bins, packed layout (several clouds back to back, sorted cloud id per point): with sorted neighbours, and for
// workspaces that do not hold the table of ball_table.hip; dense layout above 8192 points.
//
// The support array is cut into windows of 8192 or 16384 (bqb_window_shift) consecutive rows, each ordered on its
// own (curve_cells_kernel), which groups a window's points by the cell of a 16^3 grid over the
// window's bounding box; the ordering kernel also leaves where each such bin ends.  One
// wavefront serves one query: it reads which support rows belong to the query's cloud (found for
// every query by workgroups that ride along with the ordering launch), and so the windows they
// lie in, and finds in every window the bins that the cube around the ball touches - a handful
// when the radius is small against the cloud - and tests their points, 64 per step, one per
// lane.  A candidate is a hit when its squared distance is <= radius^2 and its row lies in the
// query's cloud.  The hits (at most 64) are collected in LDS, ranked by row, and written in
// ascending row order, then -1: the rows a serial scan in index order that stops after nsample
// hits (cuda/src/ball_query_gpu.cu:54-95) would have produced.
// The (window, bin) pairs of a query are walked 64 at a time.  A query whose ball touches more
// than 64 bins of one window or 512 in all, or that has more than 64 hits, is answered by that
// serial scan itself, 64 rows per step with early exit: those are the dense
// neighbourhoods, where the scan ends soon.
// ---------------------------------------------------------------------------------------
// Rows per window of the packed ball query, as a shift.  Windows of 8192 rows are ordered faster and by twice as
// many workgroups (config 4: 15 windows of 16384 rows leave most of the chip idle while they are ordered: 61 ->
// 57 us with 8192, 58 with 4096); a lane per window limits a cloud to 64 windows, so arrays above 64 x 8192 rows
// keep windows of 16384.
constexpr int BQB_SMALL_SHIFT = 13;
inline int bqb_window_shift(int64_t size_x)
{
    return size_x <= (static_cast<int64_t>(TPK_WAVE) << BQB_SMALL_SHIFT) ? BQB_SMALL_SHIFT : 14;
}
static_assert((1 << 14) == CURVE_MAX_POINTS, "the larger window is what the ordering kernel holds at most");
constexpr int BQB_HITS = TPK_WAVE; // hits a wavefront collects before it falls back to the scan
constexpr int BQB_DENSE_MIN_POINTS = 8192; // dense layout: clouds above this take the bin walk (smaller ones fit in LDS whole)
constexpr int64_t BQB_DENSE_MIN_PAIRS = 40000000; // ... when the call has at least this many (query, point) pairs

// Points per touched bin from which the bins are walked one after the other: a step of 64 candidates of one bin needs a
// third of the instructions of a step of 64 from all of them (which has to find out whose each candidate is), but a
// bin's last step is only partly filled.  300000 queries of 24 clouds (12500 points, bins of about 100): 294 us mixed,
// 266 one after the other from 48 points on, 277 from 32, 290 from 16 (the prefix sums' new last steps: 254).  Scenes
// with 4 points a bin: no difference.
constexpr int BQB_LONG_BIN = 48;

// Range of 16^3-grid cells along one axis that [v - r, v + r] can touch.  The interval is widened
// by a few ulps of its ends so that a point the fp32 radius test accepts is never left out.
__device__ __forceinline__ void bin_range(float v, float r, float lo, float scale, int& first, int& last)
{
    const float slack = (fabsf(v) + r) * 1e-6f + 1e-30f;
    first = static_cast<int>(curve_grid_cell((v - r) - slack, lo, scale) >> 2);
    last = static_cast<int>(curve_grid_cell((v + r) + slack, lo, scale) >> 2);
}

// SORTED: the nsample (<= 64) NEAREST points with squared distance < radius2, nearest first, instead of the
// first nsample in row order with squared distance <= radius2: the wavefront keeps its 64 best (distance, row)
// keys sorted across the lanes and merges the hits of a step into them (as the wavefront-per-query kernel
// further down does with the points of a cell).
// DENSE (unsorted only): the dense layout's rules instead (cuda/src/ball_query_gpu.cu:9-52) - clouds of dense_n
// consecutive rows with dense_m consecutive queries each (no cloud_rows), a hit has squared distance < radius2
// (strict), indices count from the cloud's first row, and the slots behind the last hit repeat the first hit
// (0 without any) with distance -1.
template <bool SORTED, bool DENSE>
__global__ __launch_bounds__(NG_SCAN_THREADS) void ball_query_bins_kernel(
    int size_x, int size_y, int window_shift, float radius, float radius2, int nsample, const float* __restrict__ x,
    const float* __restrict__ y, const float4* __restrict__ sorted_x, const int* __restrict__ bin_ends,
    const float4* __restrict__ grids, const int2* __restrict__ cloud_rows, int64_t* __restrict__ idx,
    float* __restrict__ dist, int dense_n, int dense_m)
{
    static_assert(!(SORTED && DENSE), "the sorted query of the dense layout has a kernel of its own");
    constexpr int WAVES = NG_SCAN_THREADS / TPK_WAVE;
    __shared__ int hit_rows[WAVES][BQB_HITS];
    __shared__ float hit_dists[WAVES][BQB_HITS];
    __shared__ int slot_rows[WAVES][TPK_WAVE]; // pair descriptors, then candidate addresses

    const int lane = threadIdx.x & (TPK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TPK_WAVE);
    const int64_t q = static_cast<int64_t>(blockIdx.x) * WAVES + wave;
    if (q >= size_y)
        return; // (no workgroup barrier anywhere in this kernel)
    int* const rows = hit_rows[wave];
    float* const dists = hit_dists[wave];
    int* const slots = slot_rows[wave];

    const float ux = y[q * 3 + 0], uy = y[q * 3 + 1], uz = y[q * 3 + 2];
    const float qx = to_vector_register(ux), qy = to_vector_register(uy), qz = to_vector_register(uz);
    int s0, s1; // the support rows of the query's cloud
    if constexpr (DENSE)
    {
        s0 = static_cast<int>(q / dense_m) * dense_n;
        s1 = s0 + dense_n;
    }
    else
    {
        const int2 cloud = cloud_rows[q];
        s0 = cloud.x;
        s1 = cloud.y;
    }
    const int64_t out = q * nsample;
    TPK_WORK_DECL

    // The walk is laid out so that dependent loads are few: all windows at once (one lane each),
    // then all (window, bin) pairs at once, then the candidates 64 at a time.
    int cnt = 0;
    // SORTED: lane i holds the i-th smallest (distance, row) key so far; a hit must beat the nsample-th
    constexpr u64 NONE = ~0ull;
    u64 best = NONE, admit = NONE;
    auto offer = [&](bool hit, float d, int row) __attribute__((always_inline)) {
        u64 cand = hit ? knn_key(d, row) : NONE;
        cand = cand < admit ? cand : NONE;
        if (__ballot(cand != NONE) == 0)
            return;
        cand = wave_sort_keys(cand, lane, true);
        best = wave_merge_ascending(best < cand ? best : cand, lane);
        admit = read_lane_key(best, nsample - 1);
    };
    const int wx0 = s0 >> window_shift;
    const int windows = s1 > s0 ? ((s1 - 1) >> window_shift) - wx0 + 1 : 0;
    bool serial = windows > TPK_WAVE; // answer by the scan in index order instead
    if (!serial && windows > 0)
    {
        // lane w: the block of bins that the ball's cube touches in window wx0 + w
        int nbins = 0, block = 0;
        if (lane < windows)
        {
            const float4 origin = grids[(wx0 + lane) * 2 + 0], scale = grids[(wx0 + lane) * 2 + 1];
            int fx, lx, fy, ly, fz, lz;
            bin_range(ux, radius, origin.x, scale.x, fx, lx);
            bin_range(uy, radius, origin.y, scale.y, fy, ly);
            bin_range(uz, radius, origin.z, scale.z, fz, lz);
            const int nx = lx - fx + 1, ny = ly - fy + 1;
            nbins = nx * ny * (lz - fz + 1);
            block = fx | (fy << 4) | (fz << 8) | ((nx - 1) << 12) | ((ny - 1) << 16) | (lane << 26);
        }
        const int pairs_before = wave_exclusive_sum(nbins);
        const int pairs = __builtin_amdgcn_readlane(pairs_before + nbins, TPK_WAVE - 1);
        // (a ball that touches more than 64 bins of one window, or 512 in all, covers so much of
        // its cloud that the scan in index order ends early)
        serial = __ballot(nbins > TPK_WAVE) != 0 || pairs > 8 * TPK_WAVE;
        // 64 (window, bin) pairs at a time; nearly always there are no more than that
        auto walk_pairs = [&](int pair0) __attribute__((always_inline)) {
            // one descriptor per pair, written by the window's lane: a window's block holds a few bins, so a loop
            // is cheaper here than the marks used for the candidates below (64.6 against 62 us on 58750 queries)
            // (What a lane reads back was written by other lanes: fences for the compiler, no instructions.  Accesses
            // through a volatile pointer were flat ones that wait for all memory: 300000 queries of 24 clouds 275 us
            // for the whole call, 264 without.)
            for (int i = max(0, pair0 - pairs_before); i < nbins && pairs_before + i < pair0 + TPK_WAVE; ++i)
                slots[pairs_before + i - pair0] = block | (i << 20);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            // lane p: where the points of pair pair0 + p start in the ordered array, and how many
            int start = 0, size = 0;
            if (pair0 + lane < pairs)
            {
                const int d = slots[lane];
                const int i = (d >> 20) & 63, window = (d >> 26) & 63;
                const int fx = d & 15, fy = (d >> 4) & 15, fz = (d >> 8) & 15;
                const int nx = ((d >> 12) & 15) + 1, ny = ((d >> 16) & 15) + 1;
                const int wx = wx0 + window;
                // (the table of the ordering kernel: 8 KiB that every wavefront reads, at home in the caches)
                // (i = ix + nx * (iy + ny * iz), taken apart by float division: exact for these small numbers)
                const int iz = static_cast<int>((static_cast<float>(i) + 0.5f) * __builtin_amdgcn_rcpf(static_cast<float>(nx * ny)));
                const int in_plane = i - iz * nx * ny;
                const int iy = static_cast<int>((static_cast<float>(in_plane) + 0.5f) * __builtin_amdgcn_rcpf(static_cast<float>(nx)));
                const int ix = in_plane - iy * nx;
                const unsigned bin = curve_bin_table.bin[(fx + ix) | ((fy + iy) << 4) | ((fz + iz) << 8)];
                const int* __restrict__ ends = bin_ends + static_cast<int64_t>(wx) * CURVE_BINS;
                start = bin ? ends[bin - 1] : 0;
                size = ends[bin] - start;
                start += wx << window_shift;
            }
            const int before = wave_exclusive_sum(size);
            const int total = __builtin_amdgcn_readlane(before + size, TPK_WAVE - 1);
            // one candidate per lane (of those that have one)
            auto test = [&](const float4 p, bool has) __attribute__((always_inline)) {
                const float d = tpk_dist2(qx, qy, qz, p.x, p.y, p.z);
                TPK_WORK_ADD(1);
                const int row = __float_as_int(p.w);
                if constexpr (SORTED)
                {
                    offer(has && d < radius2 && row >= s0 && row < s1, d, row);
                    return;
                }
                const bool hit = has && (DENSE ? d < radius2 : d <= radius2) && row >= s0 && row < s1;
                const unsigned long long mask = __ballot(hit);
                if (mask == 0)
                    return;
                const int at = cnt + static_cast<int>(tpk_prefix_count(mask));
                if (hit && at < BQB_HITS)
                {
                    rows[at] = row;
                    dists[at] = d;
                }
                cnt += __builtin_popcountll(mask);
                serial = cnt > BQB_HITS;
            };
            unsigned long long live = __ballot(size > 0);
            if (total >= BQB_LONG_BIN * __builtin_popcountll(live) && total > 0)
            {
                // Long bins: one after the other, 64 points per step, the points of a step requested a step ahead.
                int at = 0, end = 0; // (wave-uniform: what is left of the bin at hand)
                auto next_step = [&]() __attribute__((always_inline)) {
                    at += TPK_WAVE;
                    if (at < end)
                        return true;
                    if (live == 0)
                        return false;
                    const int pair = __builtin_ctzll(live);
                    live &= live - 1;
                    at = __builtin_amdgcn_readlane(start, pair);
                    end = at + __builtin_amdgcn_readlane(size, pair);
                    return true;
                };
                bool more = next_step();
                float4 ahead = sorted_x[min(at + lane, end - 1)];
                bool ahead_has = at + lane < end;
                while (more && !serial)
                {
                    const float4 p = ahead;
                    const bool has = ahead_has;
                    more = next_step();
                    if (more)
                    {
                        ahead = sorted_x[min(at + lane, end - 1)];
                        ahead_has = at + lane < end;
                    }
                    test(p, has);
                }
                return;
            }
            const int origin = start - before; // candidate c of this walk lies at origin + c, for the c of this lane's pair
            for (int c0 = 0; c0 < total && !serial; c0 += TPK_WAVE)
            {
                // Which pair does candidate c0 + lane belong to?  Every pair's lane marks the slot of its first
                // candidate in this step with its own number; a running maximum over the slots carries the
                // number on to the pair's other candidates.
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                slots[lane] = 0;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                if (size > 0 && before < c0 + TPK_WAVE && before + size > c0)
                    slots[max(before - c0, 0)] = lane;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                const int mark = slots[lane];
                const bool has = c0 + lane < total;
                const int at_x = __builtin_amdgcn_ds_bpermute(wave_inclusive_max_i32(mark) * 4, origin) + c0 + lane;
                test(sorted_x[has ? at_x : 0], has);
            }
        };
        if (!serial)
            walk_pairs(0);
        for (int pair0 = TPK_WAVE; pair0 < pairs && !serial; pair0 += TPK_WAVE)
            walk_pairs(pair0);
    }

    if constexpr (SORTED)
    {
        if (serial)
        {
            // too many windows or bins for the walk: every row of the cloud, 64 per step
            constexpr int BATCH = 4;
            for (int base = s0; base < s1; base += BATCH * TPK_WAVE)
            {
                float px[BATCH], py[BATCH], pz[BATCH];
#pragma unroll
                for (int u = 0; u < BATCH; ++u)
                {
                    const int64_t pos = min(base + u * TPK_WAVE + lane, s1 - 1);
                    px[u] = x[pos * 3 + 0];
                    py[u] = x[pos * 3 + 1];
                    pz[u] = x[pos * 3 + 2];
                }
#pragma unroll
                for (int u = 0; u < BATCH; ++u)
                {
                    const int pos = base + u * TPK_WAVE + lane;
                    const float d = tpk_dist2(qx, qy, qz, px[u], py[u], pz[u]);
                    TPK_WORK_ADD(1);
                    offer(pos < s1 && d < radius2, d, pos);
                }
            }
        }
        if (lane < nsample)
        {
            const bool found = best != NONE;
            idx[out + lane] = found ? static_cast<int64_t>(best & 0xFFFFFFFFu) : -1;
            dist[out + lane] = found ? __int_as_float(static_cast<int>(best >> 32)) : -1.0f;
        }
        TPK_WORK_FLUSH
        return;
    }
    if (!serial)
    {
        // rank of every hit among the hits (rows are distinct), then hits in order, then -1
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        const int my_row = rows[lane < cnt ? lane : 0];
        const float my_dist = dists[lane < cnt ? lane : 0];
        int rank = 0;
        for (int j = 0; j < cnt; ++j)
            rank += rows[j] < my_row ? 1 : 0;
        if (lane < cnt && rank < nsample)
        {
            idx[out + rank] = DENSE ? my_row - s0 : my_row;
            dist[out + rank] = my_dist;
        }
        int64_t filler = -1;
        if constexpr (DENSE)
        {
            // the first hit of the scan in index order = the lowest row among the hits
            const unsigned long long lowest = __ballot(lane < cnt && rank == 0);
            filler = lowest ? __shfl(my_row, __builtin_ctzll(lowest)) - s0 : 0;
        }
        for (int s = cnt + lane; s < nsample; s += TPK_WAVE)
        {
            idx[out + s] = filler;
            dist[out + s] = -1.0f;
        }
        TPK_WORK_FLUSH
        return;
    }

    ball_scan_rows<DENSE>(x, s0, s1, qx, qy, qz, radius2, nsample, lane, idx + out, dist + out TPK_WORK_ARG);
    TPK_WORK_FLUSH
}

struct GridLayout
{
    size_t sorted_a, sorted_b, boxes_a, boxes_b, wide_a, wide_b, total;
};

// Cells of a cloud of n points: ordered whole up to NG_WINDOW points, else in windows of NG_WINDOW
// consecutive points (the last one padded with cells that hold nothing).
int grid_cells(int n)
{
    return n <= NG_WINDOW ? (n + NG_CELL - 1) / NG_CELL
                          : static_cast<int>(tpk_ceil_div(n, NG_WINDOW)) * (NG_WINDOW / NG_CELL);
}
int grid_stride(int n)
{
    return n <= NG_WINDOW ? n : NG_WINDOW;
}

GridLayout grid_layout(int b, int n, int m, bool wide_first = false)
{
    auto up = [](size_t v) { return (v + 255) & ~static_cast<size_t>(255); };
    const size_t cells_a = static_cast<size_t>(grid_cells(n));
    const size_t cells_b = static_cast<size_t>(grid_cells(m));
    GridLayout l;
    size_t pos = 0;
    l.sorted_a = pos;
    pos = up(pos + static_cast<size_t>(b) * cells_a * NG_CELL * sizeof(float4));
    l.sorted_b = pos;
    pos = up(pos + static_cast<size_t>(b) * cells_b * NG_CELL * sizeof(float4));
    l.boxes_a = pos;
    pos = up(pos + static_cast<size_t>(b) * cells_a * NG_CELL_BOXES * sizeof(float4));
    l.boxes_b = pos;
    pos = up(pos + static_cast<size_t>(b) * cells_b * NG_CELL_BOXES * sizeof(float4));
    l.wide_a = l.wide_b = pos;
    if (wide_first) // (the Chamfer search: the cells of every window, wide ones first)
    {
        pos = up(pos + static_cast<size_t>(b) * cells_a * sizeof(int));
        l.wide_b = pos;
        pos = up(pos + static_cast<size_t>(b) * cells_b * sizeof(int));
    }
    l.total = pos;
    return l;
}

bool grid_supported(int b, int n, int m)
{
    // Small clouds are served as fast by the all-pairs scan; the box distances of very large ones
    // do not fit in LDS.
    return b > 0 && n >= 512 && m >= 512 && grid_cells(n) <= NG_MAX_CELLS && grid_cells(m) <= NG_MAX_CELLS;
}

} // namespace

#ifdef TPK_COUNT_WORK
extern "C" int tpk_matrix_product(int64_t count, const void* a, const void* b, float* d, void* stream)
{
    if (count < 0 || (count > 0 && (!a || !b || !d)))
        return TPK_ERR_INVALID_ARG;
    if (count == 0)
        return TPK_OK;
    if (count > (1 << 20) || ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15u))
        return TPK_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(matrix_product_kernel, dim3(static_cast<unsigned>(count)), dim3(TPK_WAVE), 0, tpk_stream(stream),
                       static_cast<const uint4*>(a), static_cast<const uint4*>(b), d);
    return tpk_launch_status();
}
#endif

size_t tpk_grid_chamfer_workspace_bytes(int b, int n, int m)
{
    return grid_supported(b, n, m) ? grid_layout(b, n, m, true).total : 0;
}

int64_t tpk_grid_chamfer_cells(int b, int n, int m)
{
    return static_cast<int64_t>(grid_cells(n) + grid_cells(m)) * b;
}

namespace {
// log2 of the wavefronts that share a cell's queries, as in three_nn's search, to fewer wavefronts: a scan on the matrix cores costs 32
// queries what it costs 16, and a wavefront's set-up is a larger part of it.  Sharing shortens the wavefronts the call would wait for, which takes
// large clouds, and is paid in wavefronts, so that few cells are shared, and in calls of many pairs fewer.  Forward, us, whole / halves / quarters:
//   512 cells of 64 queries: 1 x 16384 even 41 / 37 / 36, eight clusters 60 / 55 / 47, laser scan 226 / 130 / 92; 4 x 4096 34 / 30 / 28, 44 / 38 / 38,
//     102 / 53 / 47; 32 x 512 20.9 / 20.6 / 21.3, 21.1 / 20.6 / 21.3, 24.8 / 22.6 / 22.7
//   1024: 2 x 16384 42 / 38 / 40, 81 / 68 / 56, 227 / 130 / 101; 32 x 1024 24.5 / 25.1 / 28, 24.5 / 24.1 / 27, 32 / 29 / 31; 64 x 512 21.3 / 22.3 / 25,
//     21.2 / 21.8 / 25, 25.9 / 24.3 / 27
//   2048: 4 x 16384 44 / 44 / 52, 82 / 73 / 62, 268 / 137 / 152; 16 x 4096 34.9 / 35.7 / 41, 41 / 38 / 40, 96 / 59 / 72; 32 x 2048 31 / 33 / 37,
//     30.9 / 31.4 / 38, 49 / 46 / 58; 64 x 1024 26.9 / 29.5 / 36, 26.3 / 27.5 / 33, 36 / 34 / 40
//   4096: 8 x 16384 51 / 56 / 69, 83 / 75 / 74, 285 / 181 / 227; 32 x 4096 41 / 45 / 56, 42 / 43 / 54, 97 / 81 / 104
constexpr int64_t CHAMFER_QUARTERED_CELLS = 512, CHAMFER_HALVED_CELLS = 2048;
constexpr int64_t CHAMFER_HALVED_PAIR_CELLS = 32768; // cells times pairs of clouds: 32 pairs of 1024 cells, 16 of 2048
int chamfer_parts(int b, int n, int m)
{
    const int64_t cells = tpk_grid_chamfer_cells(b, n, m);
    return cells <= CHAMFER_QUARTERED_CELLS ? 2 : cells <= CHAMFER_HALVED_CELLS && cells * b <= CHAMFER_HALVED_PAIR_CELLS ? 1 : 0;
}
} // namespace

int tpk_grid_chamfer_fwd(int b, int n, int m, const float* xyz1, const float* xyz2, float* dist1,
                         float* dist2, int32_t* idx1, int32_t* idx2, void* workspace,
                         size_t workspace_bytes, hipStream_t s)
{
    if (!grid_supported(b, n, m) || static_cast<int64_t>(b) * 2 > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    const GridLayout l = grid_layout(b, n, m, true);
    if (!workspace || workspace_bytes < l.total || (reinterpret_cast<uintptr_t>(workspace) & 255u))
        return TPK_ERR_WORKSPACE;
    char* w = static_cast<char*>(workspace);
    PointSet a{xyz1, nullptr, static_cast<int64_t>(b) * n, n, grid_stride(n), reinterpret_cast<float4*>(w + l.sorted_a),
               reinterpret_cast<float4*>(w + l.boxes_a), nullptr, nullptr, nullptr};
    PointSet c{xyz2, nullptr, static_cast<int64_t>(b) * m, m, grid_stride(m), reinterpret_cast<float4*>(w + l.sorted_b),
               reinterpret_cast<float4*>(w + l.boxes_b), nullptr, nullptr, nullptr};
    // Both clouds' windows hold the same number of cells (clouds of one size class, the usual case): the cells
    // are handed to the wavefronts wide ones first.
    const int window_cells = set_cells(a) == set_cells(c) ? set_cells(a) : 0;
    if (window_cells > 0)
    {
        a.wide_first = reinterpret_cast<int*>(w + l.wide_a);
        c.wide_first = reinterpret_cast<int*>(w + l.wide_b);
    }
    int st = launch_curve_cells(a, c, nullptr, s);
    if (st != TPK_OK)
        return st;
    const int cells1 = grid_cells(n), cells2 = grid_cells(m);
    const int log2_parts = chamfer_parts(b, n, m);
    const int64_t waves = tpk_grid_chamfer_cells(b, n, m) << log2_parts;
    const int64_t blocks = tpk_ceil_div(waves, NG_SCAN_THREADS / TPK_WAVE);
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    const size_t lds = static_cast<size_t>(NG_SCAN_THREADS / TPK_WAVE) *
                       ((std::max(cells1, cells2) + NG_CELL - 1) / NG_CELL * NG_CELL) * sizeof(float);
    hipLaunchKernelGGL(chamfer_grid_kernel, dim3(static_cast<unsigned>(blocks)), dim3(NG_SCAN_THREADS), lds, s, n,
                       m, cells1, cells2, b, a.sorted, c.sorted, a.boxes, c.boxes, dist1, dist2, idx1, idx2, a.wide_first,
                       c.wide_first, window_cells, static_cast<int>(tpk_ceil_div(set_cells(a), curve_parts(a, c))), log2_parts);
    return tpk_launch_status();
}

// (behind the ordered copies and boxes: one word per cloud, see tpk_grid_three_nn_flags)
size_t tpk_grid_three_nn_workspace_bytes(int b, int n, int m)
{
    return grid_supported(b, n, m) ? grid_layout(b, n, m).total + ((static_cast<size_t>(b) * sizeof(int) + 255) & ~static_cast<size_t>(255)) : 0;
}

int* tpk_grid_three_nn_flags(int b, int n, int m, void* workspace, size_t workspace_bytes)
{
    const size_t need = tpk_grid_three_nn_workspace_bytes(b, n, m);
    if (!need || !workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 255u))
        return nullptr;
    return reinterpret_cast<int*>(static_cast<char*>(workspace) + grid_layout(b, n, m).total);
}

GridCells tpk_grid_three_nn_cells(int b, int n, int m, void* workspace)
{
    const GridLayout l = grid_layout(b, n, m);
    char* const w = static_cast<char*>(workspace);
    return GridCells{reinterpret_cast<float4*>(w + l.sorted_a), reinterpret_cast<float4*>(w + l.sorted_b),
                     reinterpret_cast<float4*>(w + l.boxes_b), grid_stride(n), grid_stride(m)};
}

int tpk_grid_three_nn(int b, int n, int m, const float* unknown, const float* known, float* dist2,
                      int32_t* idx, bool root, void* workspace, size_t workspace_bytes, bool flagged, bool ordered, hipStream_t s)
{
    if (!grid_supported(b, n, m) || static_cast<int64_t>(b) * 2 > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    const GridLayout l = grid_layout(b, n, m);
    if (!workspace || workspace_bytes < tpk_grid_three_nn_workspace_bytes(b, n, m) || (reinterpret_cast<uintptr_t>(workspace) & 255u))
        return TPK_ERR_WORKSPACE;
    char* w = static_cast<char*>(workspace);
    const int* only = flagged ? reinterpret_cast<const int*>(w + l.total) : nullptr;
    // (the unknown points are only queried: no boxes of their cells - the search forms the box of its 64 queries)
    const GridCells cells = tpk_grid_three_nn_cells(b, n, m, workspace);
    PointSet a{unknown, nullptr, static_cast<int64_t>(b) * n, n, cells.window_unknown, cells.sorted_unknown,
               nullptr, nullptr, nullptr, nullptr, only};
    PointSet c{known, nullptr, static_cast<int64_t>(b) * m, m, cells.window_known, cells.sorted_known,
               cells.boxes_known, nullptr, nullptr, nullptr, only};
    if (!ordered)
    {
        const int st = launch_curve_cells(a, c, nullptr, s);
        if (st != TPK_OK)
            return st;
    }
    const int qcells = grid_cells(n), ccells = grid_cells(m);
    int64_t waves = static_cast<int64_t>(qcells) * b;
    int log2_parts = 0;
    for (; log2_parts < NG_MOST_PARTS && waves * 2 <= NG_PARTED_WAVES; ++log2_parts)
        waves *= 2;
    const int64_t blocks = tpk_ceil_div(waves, NG_SCAN_THREADS / TPK_WAVE);
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    const size_t lds = static_cast<size_t>(NG_SCAN_THREADS / TPK_WAVE) * ((ccells + NG_CELL - 1) / NG_CELL * NG_CELL) *
                       sizeof(float);
    hipLaunchKernelGGL(three_nn_grid_kernel, dim3(static_cast<unsigned>(blocks)), dim3(NG_SCAN_THREADS), lds, s, n,
                       m, qcells, ccells, b, a.sorted, c.sorted, c.boxes, dist2, idx, root, only, log2_parts);
    return tpk_launch_status();
}

namespace {

// Ball query with sorted neighbours, one wavefront per query: the nsample (<= 64) nearest support
// points with squared distance < limit.  The support points lie in curve-ordered cells of 64; a
// cell whose box is out of reach is skipped; the others are tested one point per lane.  The
// wavefront keeps its 64 best (distance, index) keys sorted across the lanes: the candidates of a
// cell that beat the current nsample-th key are sorted the other way round and merged in (minimum
// per lane, then one bitonic merge).  Dense neighbourhoods - hundreds of points inside the radius -
// cost a few such merges, not an insertion per point.
// Unused slots: packed layout -1 / -1; dense layout the nearest neighbour's index (0 without any)
// and -1.  Indices are raised by index_add.
__global__ __launch_bounds__(NG_SCAN_THREADS) void ball_sorted_wave_kernel(
    int64_t queries, int n, int ccells, int nsample, float limit, bool packed, int64_t index_add,
    const float* __restrict__ query, const float4* __restrict__ sorted_support,
    const float4* __restrict__ boxes_support, const float4* __restrict__ run_boxes, float* __restrict__ dist,
    int64_t* __restrict__ idx)
{
    const int lane = threadIdx.x & (TPK_WAVE - 1);
    const int64_t q = static_cast<int64_t>(blockIdx.x) * (NG_SCAN_THREADS / TPK_WAVE) + threadIdx.x / TPK_WAVE;
    if (q >= queries)
        return; // (no workgroup barrier anywhere in this kernel)
    const int64_t cloud = q / n;
    const float4* __restrict__ cpts = sorted_support + cloud * ccells * NG_CELL;
    const float4* __restrict__ cbox = boxes_support + cloud * ccells * NG_BOX;
    const float qx = query[q * 3 + 0], qy = query[q * 3 + 1], qz = query[q * 3 + 2];

    constexpr u64 NONE = ~0ull;
    u64 best = NONE;      // lane i: the i-th smallest key so far
    u64 admit = NONE;     // the nsample-th smallest: a candidate must beat it
    float reach = limit;  // squared distance beyond which a cell cannot help
    // One cell offered to the list, one point per lane.
    auto offer = [&](int cell) __attribute__((always_inline)) {
        const float4 p = cpts[static_cast<int64_t>(cell) * NG_CELL + lane];
        const float d = tpk_dist2(qx, qy, qz, p.x, p.y, p.z);
        u64 cand = d < limit ? knn_key(d, __float_as_int(p.w)) : NONE;
        cand = cand < admit ? cand : NONE;
        if (__ballot(cand != NONE) == 0)
            return;
        cand = wave_sort_keys(cand, lane, true);
        best = wave_merge_ascending(best < cand ? best : cand, lane);
        admit = read_lane_key(best, nsample - 1);
        if (admit != NONE)
            reach = __int_as_float(static_cast<int>(admit >> 32));
    };
    if (run_boxes == nullptr)
    {
        // few cells: the box of every cell is tested, one cell per lane
        for (int first = 0; first < ccells; first += NG_CELL)
        {
            const int c = first + lane;
            const bool valid = c < ccells;
            const int cc = valid ? c : 0;
            const float lb = point_box_dist2(qx, qy, qz, cbox[cc * NG_BOX + 0], cbox[cc * NG_BOX + 1]);
            u64 live = __ballot(valid && lb * NG_MARGIN <= reach);
            while (live != 0)
            {
                const int bit = __builtin_ctzll(live);
                live &= live - 1;
                if (tpk_read_lane(lb, bit) * NG_MARGIN <= reach) // (the list may have filled up with nearer points)
                    offer(first + bit);
            }
        }
    }
    else
    {
        // Two levels: the boxes of runs of 16 consecutive cells (neighbours on the curve, so compact), one run
        // per lane; then the cells of up to four runs in reach, one cell per lane.
        const int runs = (ccells + NG_RUN - 1) / NG_RUN;
        const float4* __restrict__ rbox = run_boxes + cloud * runs * 2;
        for (int first_run = 0; first_run < runs; first_run += NG_CELL)
        {
            const int r = first_run + lane;
            const int rr = r < runs ? r : 0;
            const float run_lb = point_box_dist2(qx, qy, qz, rbox[rr * 2 + 0], rbox[rr * 2 + 1]);
            u64 live_runs = __ballot(r < runs && run_lb * NG_MARGIN <= reach);
            while (live_runs != 0)
            {
                // the next four runs in reach: lanes 16 j .. 16 j + 15 take the cells of the j-th
                int mine = -1;
#pragma unroll
                for (int j = 0; j < TPK_WAVE / NG_RUN; ++j)
                {
                    const int bit = live_runs != 0 ? __builtin_ctzll(live_runs) : -1;
                    live_runs &= live_runs - 1; // (0 stays 0)
                    mine = (lane / NG_RUN) == j ? bit : mine;
                }
                const int c = mine < 0 ? ccells : (first_run + mine) * NG_RUN + (lane % NG_RUN);
                const bool valid = c < ccells;
                const int cc = valid ? c : 0;
                const float lb = point_box_dist2(qx, qy, qz, cbox[cc * NG_BOX + 0], cbox[cc * NG_BOX + 1]);
                u64 live = __ballot(valid && lb * NG_MARGIN <= reach);
                while (live != 0)
                {
                    const int bit = __builtin_ctzll(live);
                    live &= live - 1;
                    if (tpk_read_lane(lb, bit) * NG_MARGIN > reach)
                        continue; // the list has filled up with nearer points meanwhile
                    offer(__builtin_amdgcn_readlane(c, bit));
                }
            }
        }
    }
    if (lane < nsample)
    {
        const u64 nearest = read_lane_key(best, 0);
        const bool found = best != NONE;
        const int64_t o = q * nsample + lane;
        const int64_t pad = packed ? -1 : (nearest != NONE ? static_cast<int64_t>(nearest & 0xFFFFFFFFu) + index_add : 0);
        idx[o] = found ? static_cast<int64_t>(best & 0xFFFFFFFFu) + index_add : pad;
        dist[o] = found ? __int_as_float(static_cast<int>(best >> 32)) : -1.0f;
    }
}

// Box of every run of NG_RUN consecutive cells of a cloud: (lo, hi) as two float4.
__global__ __launch_bounds__(NG_SCAN_THREADS) void run_boxes_kernel(int64_t total_runs, int runs, int ccells,
                                                                    const float4* __restrict__ boxes,
                                                                    float4* __restrict__ run_boxes)
{
    const int64_t t = static_cast<int64_t>(blockIdx.x) * NG_SCAN_THREADS + threadIdx.x;
    if (t >= total_runs)
        return;
    const int64_t cloud = t / runs;
    const int r = static_cast<int>(t - cloud * runs);
    const float4* __restrict__ cbox = boxes + cloud * ccells * NG_BOX;
    const float inf = __builtin_inff();
    float4 lo = make_float4(inf, inf, inf, 0.f), hi = make_float4(-inf, -inf, -inf, 0.f);
    // (an empty cell: lo = +inf, hi = -inf; a side that is not a number, of a cell with such a point, says nothing of the cell's others)
    auto lower = [=](float v, float side) { return side != side ? -inf : fminf(v, side); };
    auto higher = [=](float v, float side) { return side != side ? inf : fmaxf(v, side); };
    for (int c = r * NG_RUN; c < ccells && c < (r + 1) * NG_RUN; ++c)
    {
        const float4 a = cbox[c * NG_BOX + 0], b = cbox[c * NG_BOX + 1];
        lo = make_float4(lower(lo.x, a.x), lower(lo.y, a.y), lower(lo.z, a.z), 0.f);
        hi = make_float4(higher(hi.x, b.x), higher(hi.y, b.y), higher(hi.z, b.z), 0.f);
    }
    run_boxes[t * 2 + 0] = lo;
    run_boxes[t * 2 + 1] = hi;
}

struct SupportLayout
{
    size_t sorted, boxes, runs, total;
};

SupportLayout support_layout(int b, int m)
{
    auto up = [](size_t v) { return (v + 255) & ~static_cast<size_t>(255); };
    const size_t cells = static_cast<size_t>(grid_cells(m));
    SupportLayout l;
    l.sorted = 0;
    l.boxes = up(static_cast<size_t>(b) * cells * NG_CELL * sizeof(float4));
    l.runs = l.boxes + up(static_cast<size_t>(b) * cells * NG_CELL_BOXES * sizeof(float4));
    l.total = l.runs + up(static_cast<size_t>(b) * ((cells + NG_RUN - 1) / NG_RUN) * 2 * sizeof(float4));
    return l;
}

// Worth ordering the support points from this many on; below, all pairs are as fast.
bool ball_sorted_supported(int b, int m, int nsample)
{
    return b > 0 && m >= 512 && nsample >= 1 && nsample <= TPK_WAVE;
}

} // namespace

size_t tpk_grid_ball_sorted_workspace_bytes(int b, int m)
{
    return ball_sorted_supported(b, m, 1) ? support_layout(b, m).total : 0;
}

// n queries and m support points per cloud; outputs complete (padding included).
int tpk_grid_ball_sorted(int b, int n, int m, int nsample, float limit, bool packed, int64_t index_add,
                         const float* query, const float* support, float* dist, int64_t* idx, void* workspace,
                         size_t workspace_bytes, hipStream_t s)
{
    if (!ball_sorted_supported(b, m, nsample) || n < 1 || !(limit < __builtin_inff()))
        return TPK_ERR_UNSUPPORTED;
    const SupportLayout l = support_layout(b, m);
    if (!workspace || workspace_bytes < l.total || (reinterpret_cast<uintptr_t>(workspace) & 255u))
        return TPK_ERR_WORKSPACE;
    char* w = static_cast<char*>(workspace);
    PointSet none{nullptr, nullptr, 0, 1, 0, nullptr, nullptr, nullptr, nullptr};
    PointSet c{support, nullptr, static_cast<int64_t>(b) * m, m, grid_stride(m), reinterpret_cast<float4*>(w + l.sorted),
               reinterpret_cast<float4*>(w + l.boxes), nullptr, nullptr};
    int st = launch_curve_cells(none, c, nullptr, s);
    if (st != TPK_OK)
        return st;
    const int ccells = grid_cells(m), runs = (ccells + NG_RUN - 1) / NG_RUN;
    // second-level boxes pay from a few groups of 64 cells on
    float4* run_boxes = ccells > 4 * NG_CELL ? reinterpret_cast<float4*>(w + l.runs) : nullptr;
    if (run_boxes)
    {
        const int64_t total_runs = static_cast<int64_t>(b) * runs;
        hipLaunchKernelGGL(run_boxes_kernel, dim3(static_cast<unsigned>(tpk_ceil_div(total_runs, NG_SCAN_THREADS))),
                           dim3(NG_SCAN_THREADS), 0, s, total_runs, runs, ccells, c.boxes, run_boxes);
        st = tpk_launch_status();
        if (st != TPK_OK)
            return st;
    }
    const int64_t queries = static_cast<int64_t>(b) * n;
    const int64_t blocks = tpk_ceil_div(queries, NG_SCAN_THREADS / TPK_WAVE);
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(ball_sorted_wave_kernel, dim3(static_cast<unsigned>(blocks)), dim3(NG_SCAN_THREADS), 0, s, queries,
                       n, ccells, nsample, limit, packed, index_add, query, c.sorted, c.boxes, run_boxes, dist, idx);
    return tpk_launch_status();
}

size_t tpk_grid_knn_workspace_bytes(int b, int n, int m)
{
    return grid_supported(b, n, m) ? grid_layout(b, n, m).total : 0;
}

namespace {

template <int K>
int launch_knn_grid(int b, int n, int k, float limit, int qcells, int ccells, const PointSet& a, const PointSet& c,
                    float* dist2, int64_t* idx, hipStream_t s)
{
    const int64_t waves = static_cast<int64_t>(qcells) * b;
    const int64_t blocks = tpk_ceil_div(waves, NG_SCAN_THREADS / TPK_WAVE);
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    const size_t lds = static_cast<size_t>(NG_SCAN_THREADS / TPK_WAVE) * ((ccells + NG_CELL - 1) / NG_CELL * NG_CELL) *
                       sizeof(float);
    for (int first = 0; first < k; first += K)
    {
        hipLaunchKernelGGL(knn_grid_kernel<K>, dim3(static_cast<unsigned>(blocks)), dim3(NG_SCAN_THREADS), lds, s, n,
                           k, first, k - first < K ? k - first : K, limit, qcells, ccells, b, a.sorted, c.sorted, c.boxes,
                           dist2, idx);
        const int st = tpk_launch_status();
        if (st != TPK_OK)
            return st;
    }
    return TPK_OK;
}

} // namespace

// n queries and m support points per cloud.
int tpk_grid_knn(int b, int n, int m, int k, float limit, const float* query, const float* support, float* dist2,
                 int64_t* idx, void* workspace, size_t workspace_bytes, hipStream_t s)
{
    if (!grid_supported(b, n, m) || static_cast<int64_t>(b) * 2 > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    const GridLayout l = grid_layout(b, n, m);
    if (!workspace || workspace_bytes < l.total || (reinterpret_cast<uintptr_t>(workspace) & 255u))
        return TPK_ERR_WORKSPACE;
    char* w = static_cast<char*>(workspace);
    PointSet a{query, nullptr, static_cast<int64_t>(b) * n, n, grid_stride(n), reinterpret_cast<float4*>(w + l.sorted_a),
               nullptr, nullptr, nullptr};
    PointSet c{support, nullptr, static_cast<int64_t>(b) * m, m, grid_stride(m), reinterpret_cast<float4*>(w + l.sorted_b),
               reinterpret_cast<float4*>(w + l.boxes_b), nullptr, nullptr};
    int st = launch_curve_cells(a, c, nullptr, s);
    if (st != TPK_OK)
        return st;
    const int qcells = grid_cells(n), ccells = grid_cells(m);
    return launch_knn_grid<KNN_MAX_K>(b, n, k, limit, qcells, ccells, a, c, dist2, idx, s);
}

namespace {

struct BallLayout
{
    size_t sorted_x, bin_ends, grids, cloud_rows, total;
};

BallLayout ball_layout(int64_t size_x, int64_t size_y)
{
    auto up = [](size_t v) { return (v + 255) & ~static_cast<size_t>(255); };
    const size_t window = static_cast<size_t>(1) << bqb_window_shift(size_x);
    const size_t wx = (static_cast<size_t>(size_x) + window - 1) / window;
    BallLayout l;
    size_t pos = 0;
    l.sorted_x = pos;
    pos = up(pos + wx * window * sizeof(float4));
    l.bin_ends = pos;
    pos = up(pos + wx * CURVE_BINS * sizeof(int));
    l.grids = pos;
    pos = up(pos + wx * 2 * sizeof(float4));
    l.cloud_rows = pos;
    pos = up(pos + static_cast<size_t>(size_y) * sizeof(int2));
    l.total = pos;
    return l;
}

bool ball_bins_supported(int64_t size_x, int64_t size_y, int nsample)
{
    // Small problems are served as fast by the all-pairs scan; rows are 32-bit here.
    return size_x >= 8192 && size_y > 0 && nsample > 0 && size_x < (1LL << 30);
}

} // namespace

size_t tpk_grid_ball_query_workspace_bytes(int64_t size_x, int64_t size_y, int nsample)
{
    return ball_bins_supported(size_x, size_y, nsample) ? ball_layout(size_x, size_y).total : 0;
}

int tpk_grid_ball_query_partial(int64_t size_x, int64_t size_y, float radius, float radius2, int nsample, bool sorted,
                                const float* x, const float* y, const int64_t* batch_x,
                                const int64_t* batch_y, int64_t* idx, float* dist, void* workspace,
                                size_t workspace_bytes, hipStream_t s)
{
    if (!ball_bins_supported(size_x, size_y, nsample) || (sorted && nsample > TPK_WAVE))
        return TPK_ERR_UNSUPPORTED;
    const BallLayout l = ball_layout(size_x, size_y);
    if (!workspace || workspace_bytes < l.total || (reinterpret_cast<uintptr_t>(workspace) & 255u))
        return TPK_ERR_WORKSPACE;
    char* w = static_cast<char*>(workspace);
    // (cloud ids are not used for the order: bins may mix the clouds of a window, rows tell them apart)
    const int window_shift = bqb_window_shift(size_x);
    PointSet px{x, nullptr, size_x, size_x, 1 << window_shift, reinterpret_cast<float4*>(w + l.sorted_x), nullptr,
                reinterpret_cast<int*>(w + l.bin_ends), reinterpret_cast<float4*>(w + l.grids)};
    PointSet none{nullptr, nullptr, 0, 1, CURVE_MAX_POINTS, nullptr, nullptr, nullptr, nullptr};
    const CloudRows rows{batch_x, batch_y, static_cast<int>(size_x), size_y, reinterpret_cast<int2*>(w + l.cloud_rows)};
    int st = launch_curve_cells(px, none, nullptr, s, rows);
    if (st != TPK_OK)
        return st;
    constexpr int WAVES = NG_SCAN_THREADS / TPK_WAVE;
    const int64_t blocks = tpk_ceil_div(size_y, WAVES);
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    if (sorted)
        hipLaunchKernelGGL((ball_query_bins_kernel<true, false>), dim3(static_cast<unsigned>(blocks)), dim3(NG_SCAN_THREADS), 0, s,
                           static_cast<int>(size_x), static_cast<int>(size_y), window_shift, std::fabs(radius), radius2, nsample, x, y,
                           px.sorted, px.bin_ends, px.grid, rows.rows, idx, dist, 0, 0);
    else
        hipLaunchKernelGGL((ball_query_bins_kernel<false, false>), dim3(static_cast<unsigned>(blocks)), dim3(NG_SCAN_THREADS), 0, s,
                           static_cast<int>(size_x), static_cast<int>(size_y), window_shift, std::fabs(radius), radius2, nsample, x, y,
                           px.sorted, px.bin_ends, px.grid, rows.rows, idx, dist, 0, 0);
    return tpk_launch_status();
}

namespace {

// The dense layout takes the bin walk for clouds too large for the buckets of cells in LDS (ball_query.hip):
// the b clouds of n points are one array of b * n rows, cut into windows like the packed layout's.
bool ball_bins_dense_supported(int b, int n, int m, int nsample)
{
    // Ordering the points costs 17 - 30 us before the first query is answered, in which time the scan of all pairs
    // tests BQB_DENSE_MIN_PAIRS pairs: calls with fewer pairs keep the scan.  (What the host cannot know is how many
    // points a ball holds.  Where it holds hundreds, the scan in index order ends after a fraction of the cloud and
    // the walk over the bins has nothing to skip: measured 66 against 34 us for 4 x 20000 points, 5000 queries
    // each, 670 points per ball, and 222 against 162 us for 100000 points with 420 per ball - against 32 and 130 us,
    // 39 and 817 us where a ball holds a few points.)
    return n > BQB_DENSE_MIN_POINTS && b > 0 && m > 0 && nsample > 0 && static_cast<int64_t>(b) * n < (1LL << 30) &&
           static_cast<int64_t>(b) * m <= 0x7fffffffLL && static_cast<int64_t>(b) * n * m >= BQB_DENSE_MIN_PAIRS;
}

} // namespace

size_t tpk_grid_ball_query_dense_workspace_bytes(int b, int n, int m, int nsample)
{
    return ball_bins_dense_supported(b, n, m, nsample) ? ball_layout(static_cast<int64_t>(b) * n, 0).total : 0;
}

int tpk_grid_ball_query_dense(int b, int n, int m, float radius, float radius2, int nsample, const float* new_xyz,
                              const float* xyz, int64_t* idx, float* dist, void* workspace, size_t workspace_bytes,
                              hipStream_t s)
{
    if (!ball_bins_dense_supported(b, n, m, nsample))
        return TPK_ERR_UNSUPPORTED;
    const int64_t size_x = static_cast<int64_t>(b) * n, size_y = static_cast<int64_t>(b) * m;
    const BallLayout l = ball_layout(size_x, 0);
    if (!workspace || workspace_bytes < l.total || (reinterpret_cast<uintptr_t>(workspace) & 255u))
        return TPK_ERR_WORKSPACE;
    char* w = static_cast<char*>(workspace);
    const int window_shift = bqb_window_shift(size_x);
    PointSet px{xyz, nullptr, size_x, size_x, 1 << window_shift, reinterpret_cast<float4*>(w + l.sorted_x), nullptr,
                reinterpret_cast<int*>(w + l.bin_ends), reinterpret_cast<float4*>(w + l.grids)};
    PointSet none{nullptr, nullptr, 0, 1, CURVE_MAX_POINTS, nullptr, nullptr, nullptr, nullptr};
    int st = launch_curve_cells(px, none, nullptr, s);
    if (st != TPK_OK)
        return st;
    constexpr int WAVES = NG_SCAN_THREADS / TPK_WAVE;
    const int64_t blocks = tpk_ceil_div(size_y, WAVES);
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    hipLaunchKernelGGL((ball_query_bins_kernel<false, true>), dim3(static_cast<unsigned>(blocks)), dim3(NG_SCAN_THREADS), 0, s,
                       static_cast<int>(size_x), static_cast<int>(size_y), window_shift, std::fabs(radius), radius2, nsample, xyz,
                       new_xyz, px.sorted, px.bin_ends, px.grid, static_cast<const int2*>(nullptr), idx, dist, n, m);
    return tpk_launch_status();
}
