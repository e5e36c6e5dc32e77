// GRNet's two grid operators: gridding (points -> occupancy grid by trilinear weights, and its
// gradient) and cubic feature sampling (features of the grid vertices around a point, and its
// gradient).  Reference: cuda/src/gridding_gpu.cu:29-331, cuda/src/cubic_feature_sampling_gpu.cu:
// 23-210.  The reference runs one block per cloud; here every launch spreads over all points
// (or output elements) of all clouds.  Sums into the grid are formed in no fixed order, as in the
// reference (float / double atomics in memory or, for a batch, in LDS); the gridding gradient of a
// point is one thread's sum in the reference's order, so it is reproduced bit for bit.
//
// Gridding comes in two forms over the same arithmetic: the reference's native pair, which takes
// coordinates in grid units and hands the factors of every (point, vertex) from the forward to the
// backward pass, and the form of its Python front end (reference gridding.py:34-60) for a whole
// batch at once: coordinates times `factor`, points whose three products sum to zero (padding)
// left out, and a backward pass that forms the factors again from the 12 bytes of a point instead
// of reading the 128 bytes they take - of the points as the forward pass found them: it copies
// them on the way, so that a caller may change the cloud in between, as with the factors kept.
//
// Vertices outside the grid: the reference forms the linear index regardless (and writes out of
// bounds or into a neighbouring row); here such a vertex gets index -1, adds nothing to the grid
// and contributes no gradient.
#include "tpk_device.h"

#include <algorithm>
#include <cmath>

namespace {

constexpr int GR_THREADS = 256;

template <typename T>
__global__ __launch_bounds__(GR_THREADS) void fill_zero_kernel(int64_t count, T* __restrict__ out)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * GR_THREADS + threadIdx.x;
    if (i < count)
        out[i] = T(0);
}

template <typename T>
int fill_zero(int64_t count, T* out, hipStream_t s)
{
    if (count == 0)
        return TPK_OK;
    const int64_t blocks = tpk_ceil_div(count, GR_THREADS);
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(fill_zero_kernel<T>, dim3(static_cast<unsigned>(blocks)), dim3(GR_THREADS), 0, s, count, out);
    return tpk_launch_status();
}

// The two grid planes a coordinate lies between (cuda/src/gridding_gpu.cu:47-67): floor and
// ceil, the upper one raised by one when the coordinate is integral.
template <typename T>
__device__ __forceinline__ void planes(T v, int* lower, int* upper)
{
    *lower = static_cast<int>(floor(v));
    *upper = static_cast<int>(ceil(v));
    if (*lower == *upper)
        *upper += 1;
}

template <typename T>
__device__ __forceinline__ T axis_weight(T v, int plane)
{
    return T(1) - fabs(v - static_cast<T>(plane));
}

// A point in grid units and what becomes of it: the two planes per axis as offsets into the grid,
// and the factors of both.
template <typename T>
struct Trilinear
{
    int off[3][2];
    T w[3][2];
};

template <typename T>
__device__ __forceinline__ Trilinear<T> trilinear(T px, T py, T pz, float min_x, float min_y, float min_z)
{
    int plane[3][2];
    planes(px, &plane[0][0], &plane[0][1]);
    planes(py, &plane[1][0], &plane[1][1]);
    planes(pz, &plane[2][0], &plane[2][1]);
    Trilinear<T> p;
    // int - float -> float -> int, as the reference's expressions convert
#pragma unroll
    for (int side = 0; side < 2; ++side)
    {
        p.off[0][side] = static_cast<int>(plane[0][side] - min_x);
        p.off[1][side] = static_cast<int>(plane[1][side] - min_y);
        p.off[2][side] = static_cast<int>(plane[2][side] - min_z);
        p.w[0][side] = axis_weight(px, plane[0][side]);
        p.w[1][side] = axis_weight(py, plane[1][side]);
        p.w[2][side] = axis_weight(pz, plane[2][side]);
    }
    return p;
}

struct GridBox
{
    float min_x, min_y, min_z;
    int len_x, len_y, len_z;
};

template <typename T>
__device__ __forceinline__ int vertex_index(const GridBox& box, const Trilinear<T>& p, int sx, int sy, int sz)
{
    const bool inside = p.off[0][sx] >= 0 && p.off[0][sx] < box.len_x && p.off[1][sy] >= 0 && p.off[1][sy] < box.len_y &&
                        p.off[2][sz] >= 0 && p.off[2][sz] < box.len_z;
    return inside ? p.off[0][sx] * box.len_y * box.len_z + p.off[1][sy] * box.len_z + p.off[2][sz] : -1;
}

// Padding of the front end: the sum in the order torch's reduction of three values takes (first and
// third, then the second), so that the same points are left out.
template <typename T>
__device__ __forceinline__ bool is_padding(T px, T py, T pz)
{
    return (px + pz) + py == T(0);
}

// What the reference's native function returns beside the grid: vertex v = 4 * (x upper) +
// 2 * (y upper) + (z upper): LLL, LLU, LUL, LUU, ULL, ULU, UUL, UUU.
template <typename T>
__device__ __forceinline__ void store_factors(int64_t j, const GridBox& box, const Trilinear<T>& p, T* grid_pt_weights,
                                              int* grid_pt_indexes)
{
#pragma unroll
    for (int v = 0; v < 8; ++v)
    {
        const int sx = v >> 2, sy = (v >> 1) & 1, sz = v & 1;
        grid_pt_indexes[j * 8 + v] = vertex_index(box, p, sx, sy, sz);
        grid_pt_weights[j * 24 + v * 3 + 0] = p.w[0][sx];
        grid_pt_weights[j * 24 + v * 3 + 1] = p.w[1][sy];
        grid_pt_weights[j * 24 + v * 3 + 2] = p.w[2][sz];
    }
}

// What the front end's forward pass keeps of a point, as it was given.
template <typename T>
__device__ __forceinline__ void keep_point(T* kept, T x, T y, T z)
{
    kept[0] = x;
    kept[1] = y;
    kept[2] = z;
}

// cuda/src/gridding_gpu.cu:29-191.  One thread per point, sums in the zeroed grid itself: for grids
// that the kernel below cannot hold, and for more points than its LDS atomics are quick for.
template <typename T>
__global__ __launch_bounds__(GR_THREADS) void gridding_kernel(
    int64_t total_pts, int n_pts, int n_grid_vertices, GridBox box, T factor, bool drop_padding,
    const T* __restrict__ ptcloud, T* __restrict__ grid_weights, T* __restrict__ grid_pt_weights,
    int* __restrict__ grid_pt_indexes, T* __restrict__ kept)
{
    const int64_t j = static_cast<int64_t>(blockIdx.x) * GR_THREADS + threadIdx.x;
    if (j >= total_pts)
        return;
    T* grid = grid_weights + (j / n_pts) * n_grid_vertices;
    const T x = ptcloud[j * 3 + 0], y = ptcloud[j * 3 + 1], z = ptcloud[j * 3 + 2];
    if (kept)
        keep_point(kept + j * 3, x, y, z);
    const T px = x * factor, py = y * factor, pz = z * factor;
    if (drop_padding && is_padding(px, py, pz))
        return;
    const Trilinear<T> p = trilinear(px, py, pz, box.min_x, box.min_y, box.min_z);
    if (grid_pt_weights)
        store_factors(j, box, p, grid_pt_weights, grid_pt_indexes);
#pragma unroll
    for (int v = 0; v < 8; ++v)
    {
        const int sx = v >> 2, sy = (v >> 1) & 1, sz = v & 1;
        const int index = vertex_index(box, p, sx, sy, sz);
        if (index >= 0)
            atomicAdd(&grid[index], p.w[0][sx] * p.w[1][sy] * p.w[2][sz]);
    }
}

// The same sums in LDS.  A grid is dealt to `parts` workgroups (a power of two) by rows along z: the
// row of planes (ox, oy) belongs to part (3 ox + 5 oy) mod parts, so that walls, floors and other flat
// clouds spread over all of them.  A workgroup walks all points of its cloud (12 bytes each, from the
// L2), adds the vertices of its rows into LDS - a float atomic there costs 3 clocks per lane that takes
// part - and writes its rows out whole, zeros included: every element of the grid is stored once, nothing
// is filled in advance and no atomic leaves the compute unit.  Bound: the stores of the grid.
// 32 clouds of 2048 points into 64^3 grids (34 MB of grid): 42 us by fill and global atomics (0.5 M at
// 20 G/s), 13 us this way.
constexpr int GRL_THREADS = 1024;

template <typename T>
__global__ __launch_bounds__(GRL_THREADS) void gridding_lds_kernel(
    int n_pts, int parts, int rows_per_x, GridBox box, T factor, bool drop_padding, const T* __restrict__ ptcloud,
    T* __restrict__ grid_weights, T* __restrict__ grid_pt_weights, int* __restrict__ grid_pt_indexes, T* __restrict__ kept)
{
    extern __shared__ __align__(16) unsigned char gridding_lds[];
    T* sums = reinterpret_cast<T*>(gridding_lds);
    const int block = static_cast<int>(xcd_local_block(blockIdx.x, gridDim.x));
    const int cloud = block / parts, part = block - cloud * parts;
    const int shift = 31 - __builtin_clz(parts);
    const int held = box.len_x * rows_per_x * box.len_z;
    const int quads = (held * static_cast<int>(sizeof(T)) + 15) / 16; // (the LDS is a whole number of 16 bytes)
    for (int t = threadIdx.x; t < quads; t += GRL_THREADS)
        reinterpret_cast<uint4*>(gridding_lds)[t] = uint4{0, 0, 0, 0};
    __syncthreads();
    const T* points = ptcloud + static_cast<int64_t>(cloud) * n_pts * 3;
    for (int i = threadIdx.x; i < n_pts; i += GRL_THREADS)
    {
        const T x = points[static_cast<int64_t>(i) * 3 + 0], y = points[static_cast<int64_t>(i) * 3 + 1], z = points[static_cast<int64_t>(i) * 3 + 2];
        const bool stores = ((i / TPK_WAVE) & (parts - 1)) == part; // (one workgroup of the cloud's)
        if (kept && stores)
            keep_point(kept + (static_cast<int64_t>(cloud) * n_pts + i) * 3, x, y, z);
        const T px = x * factor, py = y * factor, pz = z * factor;
        if (drop_padding && is_padding(px, py, pz))
            continue;
        const Trilinear<T> p = trilinear(px, py, pz, box.min_x, box.min_y, box.min_z);
        if (grid_pt_weights && stores)
            store_factors(static_cast<int64_t>(cloud) * n_pts + i, box, p, grid_pt_weights, grid_pt_indexes);
#pragma unroll
        for (int row = 0; row < 4; ++row)
        {
            const int sx = row >> 1, sy = row & 1;
            const int ox = p.off[0][sx], oy = p.off[1][sy];
            if (ox < 0 || ox >= box.len_x || oy < 0 || oy >= box.len_y || ((3 * ox + 5 * oy) & (parts - 1)) != part)
                continue;
            T* sum = sums + (ox * rows_per_x + (oy >> shift)) * box.len_z;
            const T wxy = p.w[0][sx] * p.w[1][sy];
#pragma unroll
            for (int sz = 0; sz < 2; ++sz)
                if (p.off[2][sz] >= 0 && p.off[2][sz] < box.len_z)
                    atomicAdd(&sum[p.off[2][sz]], wxy * p.w[2][sz]);
        }
    }
    __syncthreads();
    // row k of plane ox holds oy = k * parts + (the residue that solves 3 ox + 5 oy = part mod parts)
    T* out = grid_weights + static_cast<int64_t>(cloud) * box.len_x * box.len_y * box.len_z;
    constexpr int WIDE = 16 / static_cast<int>(sizeof(T));
    const bool wide = box.len_z % WIDE == 0 && (reinterpret_cast<uintptr_t>(grid_weights) & 15) == 0;
    const int per_row = wide ? box.len_z / WIDE : box.len_z;
    for (int t = threadIdx.x; t < box.len_x * rows_per_x * per_row; t += GRL_THREADS)
    {
        const int row = t / per_row, z = t - row * per_row;
        const int ox = row / rows_per_x, k = row - ox * rows_per_x;
        const unsigned residue = (static_cast<unsigned>(part - 3 * ox) * 0xCCCCCCCDu) & static_cast<unsigned>(parts - 1); // 1 / 5
        const int oy = k * parts + static_cast<int>(residue);
        if (oy >= box.len_y)
            continue;
        const int64_t at = (static_cast<int64_t>(ox) * box.len_y + oy) * box.len_z;
        if (wide)
            reinterpret_cast<uint4*>(out + at)[z] = reinterpret_cast<const uint4*>(gridding_lds)[t];
        else
            out[at + z] = sums[t];
    }
}

// cuda/src/gridding_gpu.cu:205-305: the gradient of a point is the sum over its 8 vertices, in
// the reference's order and with its signs (upper side +, lower side -).
template <typename T>
__device__ __forceinline__ void add_vertex(T g, int v, T wx, T wy, T wz, T* gx, T* gy, T* gz)
{
    const T sx = (v >> 2) ? g : -g, sy = ((v >> 1) & 1) ? g : -g, sz = (v & 1) ? g : -g;
    *gx += sx * wy * wz;
    *gy += sy * wx * wz;
    *gz += sz * wx * wy;
}

template <typename T>
__global__ __launch_bounds__(GR_THREADS) void gridding_grad_kernel(
    int64_t total_pts, int n_pts, int n_grid_vertices, const T* __restrict__ grid_pt_weights,
    const int* __restrict__ grid_pt_indexes, const T* __restrict__ grad_grid, T* __restrict__ grad_ptcloud)
{
    const int64_t j = static_cast<int64_t>(blockIdx.x) * GR_THREADS + threadIdx.x;
    if (j >= total_pts)
        return;
    const T* grad = grad_grid + (j / n_pts) * n_grid_vertices;
    T gx = T(0), gy = T(0), gz = T(0);
#pragma unroll
    for (int v = 0; v < 8; ++v)
    {
        const int index = grid_pt_indexes[j * 8 + v];
        const T g = index >= 0 && index < n_grid_vertices ? grad[index] : T(0);
        add_vertex(g, v, grid_pt_weights[j * 24 + v * 3 + 0], grid_pt_weights[j * 24 + v * 3 + 1],
                   grid_pt_weights[j * 24 + v * 3 + 2], &gx, &gy, &gz);
    }
    grad_ptcloud[j * 3 + 0] = gx;
    grad_ptcloud[j * 3 + 1] = gy;
    grad_ptcloud[j * 3 + 2] = gz;
}

// The front end's backward pass: the factors formed again from the point, the sum above, times
// `factor`; padding takes no part in the forward pass and gets zeros.
template <typename T>
__global__ __launch_bounds__(GR_THREADS) void gridding_batch_grad_kernel(
    int64_t total_pts, int n_pts, int n_grid_vertices, GridBox box, T factor, const T* __restrict__ ptcloud,
    const T* __restrict__ grad_grid, T* __restrict__ grad_ptcloud)
{
    const int64_t j = static_cast<int64_t>(blockIdx.x) * GR_THREADS + threadIdx.x;
    if (j >= total_pts)
        return;
    const T* grad = grad_grid + (j / n_pts) * n_grid_vertices;
    const T px = ptcloud[j * 3 + 0] * factor, py = ptcloud[j * 3 + 1] * factor, pz = ptcloud[j * 3 + 2] * factor;
    T gx = T(0), gy = T(0), gz = T(0);
    if (!is_padding(px, py, pz))
    {
        const Trilinear<T> p = trilinear(px, py, pz, box.min_x, box.min_y, box.min_z);
        T g[8];
#pragma unroll
        for (int v = 0; v < 8; ++v)
        {
            const int index = vertex_index(box, p, v >> 2, (v >> 1) & 1, v & 1);
            g[v] = index >= 0 ? grad[index] : T(0);
        }
#pragma unroll
        for (int v = 0; v < 8; ++v)
            add_vertex(g[v], v, p.w[0][v >> 2], p.w[1][(v >> 1) & 1], p.w[2][v & 1], &gx, &gy, &gz);
    }
    grad_ptcloud[j * 3 + 0] = gx * factor;
    grad_ptcloud[j * 3 + 1] = gy * factor;
    grad_ptcloud[j * 3 + 2] = gz * factor;
}

// ---- cubic feature sampling: cuda/src/cubic_feature_sampling_gpu.cu:23-210 ---------------------
//
// A point's vertices are floor - (ns - 1) .. floor + ns per axis (the upper plane lies one above the
// lower one whether or not the coordinate is integral), x slowest.

// Coordinates as the front end maps them (reference cubic_feature_sampling.py:57: x * half + half), or as they are.
template <typename T>
struct CubicFrame
{
    T half;
    bool mapped;
    __device__ __forceinline__ T operator()(T v) const { return mapped ? v * half + half : v; }
};

// Vertex `v` of the point whose lower planes are (x, y, z); -1 outside the map.
__device__ __forceinline__ int cubic_vertex(int x, int y, int z, int v, int side, int scale)
{
    const int first = 1 - side / 2;
    const int vz = v % side, vy = v / side % side, vx = v / (side * side);
    const int j = x + first + vx, k = y + first + vy, m = z + first + vz;
    const bool outside = j < 0 || j >= scale || k < 0 || k >= scale || m < 0 || m >= scale;
    return outside ? -1 : (j * scale + k) * scale + m;
}

// The vertex indices of every point, for the gather below.
template <typename T>
__global__ __launch_bounds__(GR_THREADS) void cubic_indexes_kernel(int64_t total_rows, int scale, int side, int n_vertices,
                                                                   CubicFrame<T> frame, const T* __restrict__ ptcloud,
                                                                   int* __restrict__ grid_pt_indexes)
{
    const int64_t row = static_cast<int64_t>(blockIdx.x) * GR_THREADS + threadIdx.x;
    if (row >= total_rows)
        return;
    const int64_t i = row / n_vertices;
    const int x = static_cast<int>(floor(frame(ptcloud[i * 3 + 0])));
    const int y = static_cast<int>(floor(frame(ptcloud[i * 3 + 1])));
    const int z = static_cast<int>(floor(frame(ptcloud[i * 3 + 2])));
    grid_pt_indexes[row] = cubic_vertex(x, y, z, static_cast<int>(row - i * n_vertices), side, scale);
}

// Small calls: one thread per output element, channel fastest, straight from the maps - a lane's read is
// a line of its own, 1.7 clocks of a compute unit's address path each.
template <typename T>
__global__ __launch_bounds__(GR_THREADS) void cubic_gather_kernel(
    int64_t total, int n_pts, int n_vertices, int channels, int64_t cub_scale, const T* __restrict__ cubic_features,
    const int* __restrict__ grid_pt_indexes, T* __restrict__ point_features)
{
    // consecutive logical blocks (one cloud's) run on one die, whose L2 then holds that cloud's feature map
    const int64_t e = static_cast<int64_t>(xcd_local_block(blockIdx.x, gridDim.x)) * GR_THREADS + threadIdx.x;
    if (e >= total)
        return;
    const int k = static_cast<int>(e % channels);
    const int64_t pv = e / channels; // point * n_vertices + vertex, over all clouds
    const int64_t cloud = pv / (static_cast<int64_t>(n_pts) * n_vertices);
    const int vertex = grid_pt_indexes[pv];
    point_features[e] = vertex < 0 ? T(0) : cubic_features[(cloud * channels + k) * cub_scale + vertex];
}

// Otherwise the maps are turned first, (c, cells) -> (cells, c), so that what a vertex contributes is one run
// of consecutive values: the gather then reads and writes whole rows.
constexpr int CT_TILE = 64;
constexpr int CT_THREADS = 256;

// WIDE: 16 bytes per lane on both sides (cells and channels multiples of that).
template <typename T, bool WIDE>
__global__ __launch_bounds__(CT_THREADS) void cubic_turn_kernel(int channels, int64_t cub_scale, int cell_tiles, int channel_tiles,
                                                                const T* __restrict__ maps, T* __restrict__ turned)
{
    constexpr int V = WIDE ? 16 / static_cast<int>(sizeof(T)) : 1;
    __shared__ T tile[CT_TILE][CT_TILE + 1];
    const unsigned block = xcd_local_block(blockIdx.x, gridDim.x);
    const int channel_tile = static_cast<int>(block % channel_tiles);
    const unsigned rest = block / channel_tiles;
    const int64_t cell0 = static_cast<int64_t>(rest % cell_tiles) * CT_TILE;
    const int64_t cloud = rest / cell_tiles;
    const int c0 = channel_tile * CT_TILE;
    const T* from = maps + cloud * channels * cub_scale;
    T* to = turned + cloud * channels * cub_scale;
    constexpr int ACROSS = CT_TILE / V, STEP = CT_THREADS / ACROSS;
    const int x = threadIdx.x % ACROSS * V, y = threadIdx.x / ACROSS;
    struct alignas(sizeof(T) * V) Piece
    {
        T v[V];
    };
    Piece piece[CT_TILE / STEP];
#pragma unroll
    for (int r = 0; r < CT_TILE; r += STEP)
        if (c0 + y + r < channels && cell0 + x < cub_scale)
            piece[r / STEP] = *reinterpret_cast<const Piece*>(from + static_cast<int64_t>(c0 + y + r) * cub_scale + cell0 + x);
#pragma unroll
    for (int r = 0; r < CT_TILE; r += STEP)
#pragma unroll
        for (int i = 0; i < V; ++i)
            tile[y + r][x + i] = piece[r / STEP].v[i];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < CT_TILE; r += STEP)
        if (cell0 + y + r < cub_scale && c0 + x < channels)
        {
            Piece out;
#pragma unroll
            for (int i = 0; i < V; ++i)
                out.v[i] = tile[x + i][y + r];
            *reinterpret_cast<Piece*>(to + (cell0 + y + r) * channels + c0 + x) = out;
        }
}

// A workgroup finds the vertices of its rows once, in LDS, and copies: bound by the stores of the rows, which
// pass the caches by so that these hold the turned maps.  V: what a lane copies at a time (16 bytes where the
// channels are a multiple of that); magic: 2^32 / per_row rounded up.
constexpr int CR_ROWS = 256; // at most, per workgroup

template <typename T, typename V>
__global__ __launch_bounds__(GR_THREADS) void cubic_rows_kernel(int64_t total_rows, int rows_per_block, int n_pts, int n_vertices, int side,
                                                                unsigned per_row, unsigned magic, int scale, CubicFrame<T> frame,
                                                                const T* __restrict__ ptcloud, const V* __restrict__ turned,
                                                                V* __restrict__ point_features, int* __restrict__ grid_pt_indexes)
{
    __shared__ int64_t from[CR_ROWS]; // first element of the row's source, -1: zeros
    const int64_t row0 = static_cast<int64_t>(xcd_local_block(blockIdx.x, gridDim.x)) * rows_per_block;
    const int rows = static_cast<int>(tpk_min64(rows_per_block, total_rows - row0));
    const int64_t cub_scale = static_cast<int64_t>(scale) * scale * scale;
    if (static_cast<int>(threadIdx.x) < rows)
    {
        const int64_t row = row0 + threadIdx.x, i = row / n_vertices;
        const int x = static_cast<int>(floor(frame(ptcloud[i * 3 + 0])));
        const int y = static_cast<int>(floor(frame(ptcloud[i * 3 + 1])));
        const int z = static_cast<int>(floor(frame(ptcloud[i * 3 + 2])));
        const int vertex = cubic_vertex(x, y, z, static_cast<int>(row - i * n_vertices), side, scale);
        grid_pt_indexes[row] = vertex;
        from[threadIdx.x] = vertex < 0 ? -1 : (i / n_pts * cub_scale + vertex) * per_row;
    }
    __syncthreads();
    V* out = point_features + row0 * per_row;
    const unsigned pieces = static_cast<unsigned>(rows) * per_row;
    constexpr unsigned UNROLL = 8;
    for (unsigned first = threadIdx.x; first < pieces; first += UNROLL * GR_THREADS)
    {
        V value[UNROLL];
#pragma unroll
        for (unsigned u = 0; u < UNROLL; ++u)
        {
            const unsigned e = first + u * GR_THREADS;
            value[u] = V{};
            if (e < pieces)
            {
                const unsigned row = per_row == 1 ? e : __umulhi(e, magic);
                const int64_t at = from[row];
                if (at >= 0)
                    value[u] = turned[at + (e - row * per_row)];
            }
        }
#pragma unroll
        for (unsigned u = 0; u < UNROLL; ++u)
            if (first + u * GR_THREADS < pieces)
                __builtin_nontemporal_store(value[u], &out[first + u * GR_THREADS]);
    }
}

// cuda/src/cubic_feature_sampling_gpu.cu:138-175 as the reference's scatter, one atomic per term, in no fixed order: what
// neither of the two kernels below takes.
template <typename T>
__global__ __launch_bounds__(GR_THREADS) void cubic_scatter_kernel(
    int64_t total, int n_pts, int n_vertices, int channels, int64_t cub_scale,
    const T* __restrict__ grad_point_features, const int* __restrict__ grid_pt_indexes,
    T* __restrict__ grad_cubic_features)
{
    const int64_t e = static_cast<int64_t>(blockIdx.x) * GR_THREADS + threadIdx.x;
    if (e >= total)
        return;
    const int k = static_cast<int>(e % channels);
    const int64_t pv = e / channels;
    const int64_t cloud = pv / (static_cast<int64_t>(n_pts) * n_vertices);
    const int vertex = grid_pt_indexes[pv];
    if (vertex >= 0 && vertex < cub_scale)
        atomicAdd(&grad_cubic_features[(cloud * channels + k) * cub_scale + vertex], grad_point_features[e]);
}

// The same sums in LDS: a workgroup owns `group` channels of one cloud's maps (group * scale^3 sums), walks all entries of
// the cloud, adds its channels' terms with LDS atomics and writes the maps out in order.  Bound: the atomics, 1.3 ns of a
// compute unit per term (3 clocks), where one in memory costs the chip 24 ps.
constexpr int CS_THREADS = 1024;
constexpr int64_t CS_BYTES = 128 * 1024; // sums per workgroup at most

template <typename T>
__global__ __launch_bounds__(CS_THREADS) void cubic_scatter_lds_kernel(
    int n_pts, int n_vertices, int channels, int group, int64_t cub_scale, const T* __restrict__ grad_point_features,
    const int* __restrict__ grid_pt_indexes, T* __restrict__ grad_cubic_features)
{
    extern __shared__ __align__(16) unsigned char cubic_lds[];
    T* sums = reinterpret_cast<T*>(cubic_lds);
    // the workgroups of one cloud read the same lines of the gradient (each its own channels): they
    // are kept on one die, so that one L2 serves them
    const int groups = (channels + group - 1) / group;
    const int block = static_cast<int>(xcd_local_block(blockIdx.x, gridDim.x));
    const int cloud = block / groups;
    const int k0 = (block - cloud * groups) * group;
    const int width = min(group, channels - k0);
    const int64_t cells = static_cast<int64_t>(width) * cub_scale;
    for (int64_t t = threadIdx.x; t < cells; t += CS_THREADS)
        sums[t] = T(0);
    __syncthreads();
    const int64_t entries = static_cast<int64_t>(n_pts) * n_vertices;
    const int* indexes = grid_pt_indexes + cloud * entries;
    const T* grads = grad_point_features + cloud * entries * channels;
    // consecutive threads take the channels of one entry, then the next entry
    for (int64_t t = threadIdx.x; t < entries * width; t += CS_THREADS)
    {
        const int64_t entry = t / width;
        const int k = static_cast<int>(t - entry * width);
        const int vertex = indexes[entry];
        if (vertex >= 0 && vertex < cub_scale)
            atomicAdd(&sums[k * cub_scale + vertex], grads[entry * channels + k0 + k]);
    }
    __syncthreads();
    T* out = grad_cubic_features + (static_cast<int64_t>(cloud) * channels + k0) * cub_scale;
    for (int64_t t = threadIdx.x; t < cells; t += CS_THREADS)
        out[t] = sums[t];
}

// The gradient of the maps as a gather.  A workgroup owns a span of cells of one cloud: it sorts the cloud's
// (point, vertex) entries that lie in the span by cell (counting sort in LDS, the indices come from the L2),
// then walks the sorted list - equal runs of it per group of LANES lanes, a lane per channel, the rows of
// the gradient coming in as whole lines, 16 in flight - adds up while the cell stays the same and puts a
// finished sum into LDS; what runs share at their ends is added there atomically.  The span leaves as whole lines
// per channel.  (One pass that keeps the indices in registers between counting and placing spills: 52 us; three
// 32-bit divisions per index instead of masks, and entries handled lane by lane instead of in scalars: 59 us.)
// Every row of the gradient is read once and every element of the maps written once, where
// sums by LDS atomics (194 clocks per 64 terms) bounded the version before: 32 clouds of 2048 points, 64
// channels, 16^3 cells 219 us, 44 us this way.  Bound: the stream of gradient rows.
constexpr int CB_THREADS = 1024;
constexpr int CB_LIST = 2048;   // entries sorted at a time
constexpr int CB_CHANNELS = 64; // channels summed at a time
constexpr int CB_LINE = 16;     // cells that stay together: 64 bytes of a channel

template <typename T>
struct CubicSpan
{
    static constexpr int CELLS = sizeof(T) == 4 ? 256 : 128; // (two workgroups per compute unit)
    T sums[CELLS][CB_CHANNELS + 1];
    unsigned entry[CB_LIST];
    unsigned short cell[CB_LIST];
    int count[CELLS + 1];
    int total;
};

// (float32, a lane per channel: two workgroups per compute unit, 8 wavefronts per SIMD; the other forms need the
// registers of one)
template <typename T, int LANES>
__global__ __launch_bounds__(CB_THREADS, sizeof(T) == 4 && LANES == TPK_WAVE ? 8 : 4) void cubic_spans_kernel(
                                                                 int n_pts, int n_vertices, int channels, int64_t cub_scale, int spans,
                                                                 const T* __restrict__ grad_point_features,
                                                                 const int* __restrict__ grid_pt_indexes,
                                                                 T* __restrict__ grad_cubic_features)
{
    extern __shared__ __align__(16) unsigned char cubic_lds[];
    CubicSpan<T>& lds = *reinterpret_cast<CubicSpan<T>*>(cubic_lds);
    constexpr int CELLS = CubicSpan<T>::CELLS;
    const int block = static_cast<int>(xcd_local_block(blockIdx.x, gridDim.x));
    const int cloud = block / spans;
    const int span = block - cloud * spans, span_bits = 31 - __builtin_clz(spans); // (a power of two)
    // Cell c lies in line c / LINE; lines are dealt out spans at a time, every turn starting one span further on, so
    // that no plane of the map - where a flat cloud's points would be - falls to one workgroup.
    const unsigned lines = static_cast<unsigned>((cub_scale + CB_LINE - 1) / CB_LINE);
    const int cells = static_cast<int>((lines + spans - 1) / spans) * CB_LINE; // places, some beyond the map
    const int64_t entries = static_cast<int64_t>(n_pts) * n_vertices;
    const int* indexes = grid_pt_indexes + cloud * entries;
    const T* grads = grad_point_features + cloud * entries * channels;
    constexpr int WALKERS = CB_THREADS / LANES;
    const int walker = threadIdx.x / LANES, lane = threadIdx.x % LANES;

    // the span's entries among [begin, end): f(entry, cell of the span); BATCH indices per thread on their way at a time
    auto own_entries = [&](int64_t begin, int64_t end, auto&& f) {
        constexpr int BATCH = 8;
        for (; begin < end; begin += BATCH * CB_THREADS)
        {
            const int* from = indexes + begin;
            const int length = static_cast<int>(tpk_min64(end - begin, BATCH * CB_THREADS));
            unsigned index[BATCH];
#pragma unroll
            for (int i = 0; i < BATCH; ++i)
                index[i] = static_cast<int>(threadIdx.x) < length - i * CB_THREADS ? (from + i * CB_THREADS)[threadIdx.x] : -1;
#pragma unroll
            for (int i = 0; i < BATCH; ++i)
            {
                const unsigned line = index[i] / CB_LINE, turn = line >> span_bits;
                if (index[i] < static_cast<unsigned>(cub_scale) && ((line + turn) & (spans - 1)) == static_cast<unsigned>(span))
                    f(begin + threadIdx.x + i * CB_THREADS, static_cast<int>(turn * CB_LINE + index[i] % CB_LINE));
            }
        }
    };
    auto count = [&](int64_t begin, int64_t end) {
        __syncthreads();
        for (int t = threadIdx.x; t < CELLS; t += CB_THREADS)
            lds.count[t] = 0;
        __syncthreads();
        own_entries(begin, end, [&](int64_t, int c) { atomicAdd(&lds.count[c], 1); });
        __syncthreads();
        if (threadIdx.x < TPK_WAVE)
        {
            int before = 0;
            for (int at = 0; at < CELLS; at += TPK_WAVE)
            {
                const int v = lds.count[at + threadIdx.x];
                const int ahead = wave_exclusive_sum(v);
                lds.count[at + threadIdx.x] = before + ahead;
                before += tpk_read_lane(ahead + v, TPK_WAVE - 1);
            }
            if (threadIdx.x == 0)
                lds.total = before;
        }
        __syncthreads();
        return lds.total;
    };

    for (int c0 = 0; c0 < channels; c0 += CB_CHANNELS)
    {
        const int width = min(CB_CHANNELS, channels - c0);
        for (int t = threadIdx.x; t < CELLS * (CB_CHANNELS + 1); t += CB_THREADS)
            (&lds.sums[0][0])[t] = T(0);
        int64_t begin = 0, size = entries;
        while (begin < entries)
        {
            int64_t end = tpk_min64(begin + size, entries);
            int have = count(begin, end);
            while (have > CB_LIST)
            {
                // fewer entries at a time: what should give three quarters of a list, in any case no more than a list
                size = tpk_min64(size / 2, size * (3 * CB_LIST / 4) / have);
                size = size < CB_LIST ? CB_LIST : size;
                end = tpk_min64(begin + size, entries);
                have = count(begin, end);
            }
            own_entries(begin, end, [&](int64_t e, int c) {
                const int at = atomicAdd(&lds.count[c], 1);
                lds.entry[at] = static_cast<unsigned>(e - begin);
                lds.cell[at] = static_cast<unsigned short>(c);
            });
            __syncthreads();
            // Runs end where a cell ends, if that is not far: a sum that two runs share goes through an LDS atomic, 192
            // clocks for 64 lanes.  (LANES = 64: what follows is the same for a wavefront's lanes and kept in scalars;
            // the walk is bound by instruction issue.)
            auto same_for_group = [&](int v) { return LANES == TPK_WAVE ? __builtin_amdgcn_readfirstlane(v) : v; };
            auto run_start = [&](int w) {
                const int even = static_cast<int>(static_cast<int64_t>(have) * w / WALKERS);
                for (int q = even; q < even + 32; ++q)
                    if (q == 0 || q >= have || lds.cell[q] != lds.cell[q - 1])
                        return q < have ? q : have;
                return even;
            };
            const int q0 = same_for_group(run_start(walker)), q1 = same_for_group(run_start(walker + 1));
            int shared_start = same_for_group(q0 > 0 && q0 < q1 && lds.cell[q0] == lds.cell[q0 - 1]);
            const int shared_end = same_for_group(q1 > q0 && q1 < have && lds.cell[q1] == lds.cell[q1 - 1]);
            // (lanes beyond the channels go along: theirs are entries of the list too)
            const char* column = reinterpret_cast<const char*>(grads + begin * channels + c0 + min(lane, width - 1));
            const unsigned row_bytes = static_cast<unsigned>(channels) * static_cast<unsigned>(sizeof(T));
            int open = same_for_group(q0 < q1 ? lds.cell[q0] : 0);
            T sum = T(0);
            auto put = [&](int shared) {
                if (lane >= width)
                    return;
                if (shared)
                    atomicAdd(&lds.sums[open][lane], sum);
                else
                    lds.sums[open][lane] += sum;
            };
            // A group takes up its entries a lane each; rows are asked for AHEAD entries before they are added.
            constexpr int AHEAD = sizeof(T) == 4 ? 16 : 8;
            for (int q = q0; q < q1; q += LANES)
            {
                const int n = min(LANES, q1 - q);
                // (beyond the end: the last entry again, to a cell that is none - no branch around a load, behind one the
                // compiler waits for all loads in flight)
                const int mine = q + min(lane, n - 1);
                const int my_offset = static_cast<int>(lds.entry[mine] * row_bytes);
                const int my_cell = lds.cell[mine];
                auto of = [&](int v, int i) {
                    i = min(i, LANES - 1);
                    return LANES == TPK_WAVE ? __builtin_amdgcn_readlane(v, i) : __shfl(v, i, LANES);
                };
                auto row = [&](int i) { return *reinterpret_cast<const T*>(column + static_cast<unsigned>(of(my_offset, i))); };
                T value[AHEAD];
#pragma unroll
                for (int a = 0; a < AHEAD; ++a)
                    value[a] = row(a);
                for (int first = 0; first < n; first += AHEAD)
#pragma unroll
                    for (int a = 0; a < AHEAD; ++a)
                    {
                        const T v = value[a];
                        value[a] = row(first + a + AHEAD);
                        if (first + a < n)
                        {
                            const int c = of(my_cell, first + a);
                            if (c != open)
                            {
                                put(shared_start);
                                shared_start = 0;
                                open = c;
                                sum = T(0);
                            }
                            sum += v;
                        }
                    }
            }
            if (q0 < q1)
                put(shared_start | shared_end);
            begin = end;
        }
        __syncthreads();
        T* out = grad_cubic_features + (static_cast<int64_t>(cloud) * channels + c0) * cub_scale;
        const int place = threadIdx.x % CELLS; // (the same in every turn of the loop)
        const unsigned turn = place / CB_LINE, line = turn * spans + ((span - turn) & (spans - 1));
        const int64_t c = static_cast<int64_t>(line) * CB_LINE + place % CB_LINE;
        if (place < cells && c < cub_scale)
            for (int k = threadIdx.x / CELLS; k < width; k += CB_THREADS / CELLS)
                out[k * cub_scale + c] = lds.sums[place][k];
        __syncthreads();
    }
}

// How many workgroups share a grid in gridding_lds_kernel, and their LDS; 0: take gridding_kernel.
// At most 64 KiB of sums per workgroup where rows allow it (two of 1024 threads per compute unit, one
// adding while the other stores), more parts until every compute unit has one; the 8 n / parts atomics of
// a workgroup cost 3 clocks each, so beyond 4096 points per part (40 us) the global atomics of the other
// kernel - which spread over the chip whatever the number of clouds - are quicker.
template <typename T>
int gridding_parts(int b, int n_pts, const GridBox& box, int* rows_per_x, size_t* lds)
{
    int parts = 1;
    auto bytes = [&](int p) { return static_cast<int64_t>(box.len_x) * tpk_ceil_div(box.len_y, p) * box.len_z * static_cast<int64_t>(sizeof(T)); };
    while (parts < box.len_y && bytes(parts) > 64 * 1024)
        parts *= 2;
    while (parts < box.len_y && parts < 4096 && (static_cast<int64_t>(b) * parts < TPK_COMPUTE_UNITS || n_pts / parts > 4096) &&
           bytes(parts) > 8 * 1024)
        parts *= 2;
    if (bytes(parts) > 128 * 1024 || n_pts / parts > 4096 || static_cast<int64_t>(b) * parts > 0x7fffffffLL)
        return 0;
    *rows_per_x = static_cast<int>(tpk_ceil_div(box.len_y, parts));
    *lds = static_cast<size_t>(tpk_ceil_div(bytes(parts), 16) * 16);
    return parts;
}

bool grid_box(float min_x, float max_x, float min_y, float max_y, float min_z, float max_z, GridBox* box)
{
    // cuda/src/gridding_gpu.cu:199-202
    const int len_x = static_cast<int>(max_x - min_x + 1), len_y = static_cast<int>(max_y - min_y + 1);
    const int len_z = static_cast<int>(max_z - min_z + 1);
    *box = GridBox{min_x, min_y, min_z, len_x, len_y, len_z};
    return len_x > 0 && len_y > 0 && len_z > 0;
}

template <typename T>
int gridding_fwd(int b, int n_pts, const GridBox& box, T factor, bool drop_padding, const T* ptcloud, T* grid_weights,
                 T* grid_pt_weights, int32_t* grid_pt_indexes, T* kept, hipStream_t s)
{
    const int64_t vertices = static_cast<int64_t>(box.len_x) * box.len_y * box.len_z;
    if (vertices > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    if (b == 0)
        return TPK_OK;
    int rows_per_x = 0;
    size_t lds = 0;
    const int parts = n_pts > 0 ? gridding_parts<T>(b, n_pts, box, &rows_per_x, &lds) : 0;
    if (parts > 0)
    {
        const int allowed = tpk_allow_lds(reinterpret_cast<const void*>(gridding_lds_kernel<T>), lds);
        if (allowed != TPK_OK)
            return allowed;
        hipLaunchKernelGGL(gridding_lds_kernel<T>, dim3(static_cast<unsigned>(b) * parts), dim3(GRL_THREADS), lds, s, n_pts,
                           parts, rows_per_x, box, factor, drop_padding, ptcloud, grid_weights, grid_pt_weights,
                           grid_pt_indexes, kept);
        return tpk_launch_status();
    }
    int st = fill_zero<T>(static_cast<int64_t>(b) * vertices, grid_weights, s);
    if (st != TPK_OK || n_pts == 0)
        return st;
    const int64_t total = static_cast<int64_t>(b) * n_pts;
    const int64_t blocks = tpk_ceil_div(total, GR_THREADS);
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(gridding_kernel<T>, dim3(static_cast<unsigned>(blocks)), dim3(GR_THREADS), 0, s, total, n_pts,
                       static_cast<int>(vertices), box, factor, drop_padding, ptcloud, grid_weights, grid_pt_weights,
                       grid_pt_indexes, kept);
    return tpk_launch_status();
}

// The reference's native function: coordinates in grid units, factors and vertices returned.
template <typename T>
int gridding_native(int b, int n_pts, float min_x, float max_x, float min_y, float max_y, float min_z, float max_z,
                    const T* ptcloud, T* grid_weights, T* grid_pt_weights, int32_t* grid_pt_indexes, hipStream_t s)
{
    GridBox box;
    if (b < 0 || n_pts < 0 || !grid_box(min_x, max_x, min_y, max_y, min_z, max_z, &box))
        return TPK_ERR_INVALID_ARG;
    if (b > 0 && (!grid_weights || (n_pts > 0 && (!ptcloud || !grid_pt_weights || !grid_pt_indexes))))
        return TPK_ERR_INVALID_ARG;
    return gridding_fwd<T>(b, n_pts, box, T(1), false, ptcloud, grid_weights, grid_pt_weights, grid_pt_indexes, nullptr, s);
}

// The front end: a grid over [-scale, scale - 1] per axis, coordinates times `scale`.
template <typename T>
int gridding_batch(int b, int n_pts, double scale, const T* ptcloud, T* grid_weights, T* kept, hipStream_t s)
{
    GridBox box;
    const float lo = static_cast<float>(-scale), hi = static_cast<float>(scale - 1);
    if (b < 0 || n_pts < 0 || !grid_box(lo, hi, lo, hi, lo, hi, &box))
        return TPK_ERR_INVALID_ARG;
    if (b > 0 && (!grid_weights || (n_pts > 0 && !ptcloud)))
        return TPK_ERR_INVALID_ARG;
    return gridding_fwd<T>(b, n_pts, box, static_cast<T>(scale), true, ptcloud, grid_weights, nullptr, nullptr, kept, s);
}

template <typename T>
int gridding_batch_grad(int b, int n_pts, double scale, const T* ptcloud, const T* grad_grid, T* grad_ptcloud, hipStream_t s)
{
    GridBox box;
    const float lo = static_cast<float>(-scale), hi = static_cast<float>(scale - 1);
    if (b < 0 || n_pts < 0 || !grid_box(lo, hi, lo, hi, lo, hi, &box))
        return TPK_ERR_INVALID_ARG;
    if (b == 0 || n_pts == 0)
        return TPK_OK;
    if (!ptcloud || !grad_grid || !grad_ptcloud)
        return TPK_ERR_INVALID_ARG;
    const int64_t vertices = static_cast<int64_t>(box.len_x) * box.len_y * box.len_z;
    const int64_t total = static_cast<int64_t>(b) * n_pts;
    const int64_t blocks = tpk_ceil_div(total, GR_THREADS);
    if (vertices > 0x7fffffffLL || blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(gridding_batch_grad_kernel<T>, dim3(static_cast<unsigned>(blocks)), dim3(GR_THREADS), 0, s, total,
                       n_pts, static_cast<int>(vertices), box, static_cast<T>(scale), ptcloud, grad_grid, grad_ptcloud);
    return tpk_launch_status();
}

template <typename T>
int gridding_bwd(int b, int n_pts, int n_grid_vertices, const T* grid_pt_weights, const int32_t* grid_pt_indexes,
                 const T* grad_grid, T* grad_ptcloud, hipStream_t s)
{
    if (b < 0 || n_pts < 0 || n_grid_vertices < 0)
        return TPK_ERR_INVALID_ARG;
    if (b == 0 || n_pts == 0)
        return TPK_OK;
    if (!grid_pt_weights || !grid_pt_indexes || !grad_ptcloud || (n_grid_vertices > 0 && !grad_grid))
        return TPK_ERR_INVALID_ARG;
    const int64_t total = static_cast<int64_t>(b) * n_pts;
    const int64_t blocks = tpk_ceil_div(total, GR_THREADS);
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(gridding_grad_kernel<T>, dim3(static_cast<unsigned>(blocks)), dim3(GR_THREADS), 0, s, total,
                       n_pts, n_grid_vertices, grid_pt_weights, grid_pt_indexes, grad_grid, grad_ptcloud);
    return tpk_launch_status();
}

// (2 * neighborhood_size)^3, or -1 when that does not fit
int64_t cubic_vertices(int neighborhood_size)
{
    if (neighborhood_size < 1 || neighborhood_size > 64)
        return -1;
    const int64_t side = 2 * static_cast<int64_t>(neighborhood_size);
    return side * side * side;
}

// Whether the maps are turned first: an element gathered from them as they are costs 2.8 ps, from turned ones 0.7 ps,
// turning 1.6 ps per element of the maps and a launch.
bool cubic_turns(int b, int n_pts, int channels, int scale, int64_t nv)
{
    const double per_cell = static_cast<double>(b) * channels;
    const double rows = per_cell * n_pts * static_cast<double>(nv), cells = per_cell * scale * static_cast<double>(scale) * scale;
    return rows > 0.8 * cells + 1.5e6 && cells < 2.0e9 && channels < 65536;
}

template <typename T>
int cubic_fwd(int b, int n_pts, int channels, int scale, int neighborhood_size, bool mapped, const T* ptcloud,
              const T* cubic_features, T* point_features, int32_t* grid_pt_indexes, void* workspace, size_t workspace_bytes,
              hipStream_t s)
{
    const int64_t nv = cubic_vertices(neighborhood_size);
    if (b < 0 || n_pts < 0 || channels < 0 || scale <= 0 || nv < 0 || scale > 1290)
        return TPK_ERR_INVALID_ARG;
    if (b == 0 || n_pts == 0)
        return TPK_OK;
    if (!ptcloud || !grid_pt_indexes || (channels > 0 && (!cubic_features || !point_features)))
        return TPK_ERR_INVALID_ARG;
    const int64_t total_rows = static_cast<int64_t>(b) * n_pts * nv;
    const int64_t total = total_rows * channels;
    const int64_t blocks_rows = tpk_ceil_div(total_rows, GR_THREADS), blocks = tpk_ceil_div(total, GR_THREADS);
    if (blocks > 0x7fffffffLL || blocks_rows > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    const int side = 2 * neighborhood_size, vertices = static_cast<int>(nv);
    const int64_t cub = static_cast<int64_t>(scale) * scale * scale;
    const CubicFrame<T> frame{static_cast<T>(scale / 2.0), mapped};
    if (total > 0 && workspace && cubic_turns(b, n_pts, channels, scale, nv))
    {
        if (workspace_bytes < static_cast<size_t>(b * channels * cub) * sizeof(T) || (reinterpret_cast<uintptr_t>(workspace) & 15) != 0)
            return TPK_ERR_WORKSPACE;
        const int64_t cell_tiles = tpk_ceil_div(cub, CT_TILE), channel_tiles = tpk_ceil_div(channels, CT_TILE);
        const int64_t tiles = cell_tiles * channel_tiles * b;
        if (tiles > 0x7fffffffLL)
            return TPK_ERR_UNSUPPORTED;
        T* turned = static_cast<T*>(workspace);
        constexpr int WIDE = 16 / static_cast<int>(sizeof(T));
        typedef unsigned Quad __attribute__((ext_vector_type(4)));
        const bool wide = channels % WIDE == 0 && ((reinterpret_cast<uintptr_t>(point_features) | reinterpret_cast<uintptr_t>(cubic_features)) & 15) == 0;
        const auto turn = wide && cub % WIDE == 0 ? cubic_turn_kernel<T, true> : cubic_turn_kernel<T, false>;
        hipLaunchKernelGGL(turn, dim3(static_cast<unsigned>(tiles)), dim3(CT_THREADS), 0, s, channels, cub,
                           static_cast<int>(cell_tiles), static_cast<int>(channel_tiles), cubic_features, turned);
        const int per_row = wide ? channels / WIDE : channels;
        // (about 4096 pieces per workgroup; below 2^16, where the multiplication by `magic` is exact)
        const int rows = per_row >= 4096 ? 1 : 4096 / per_row > CR_ROWS ? CR_ROWS : 4096 / per_row;
        if (static_cast<int64_t>(rows) * per_row >= 65536)
            return TPK_ERR_UNSUPPORTED;
        const unsigned magic = static_cast<unsigned>(((uint64_t(1) << 32) + per_row - 1) / per_row);
        const unsigned grid = static_cast<unsigned>(tpk_ceil_div(total_rows, rows));
        if (wide)
            hipLaunchKernelGGL((cubic_rows_kernel<T, Quad>), dim3(grid), dim3(GR_THREADS), 0, s, total_rows, rows, n_pts, vertices, side,
                               static_cast<unsigned>(per_row), magic, scale, frame, ptcloud, reinterpret_cast<const Quad*>(turned),
                               reinterpret_cast<Quad*>(point_features), grid_pt_indexes);
        else
            hipLaunchKernelGGL((cubic_rows_kernel<T, T>), dim3(grid), dim3(GR_THREADS), 0, s, total_rows, rows, n_pts, vertices, side,
                               static_cast<unsigned>(per_row), magic, scale, frame, ptcloud, turned, point_features, grid_pt_indexes);
        return tpk_launch_status();
    }
    hipLaunchKernelGGL(cubic_indexes_kernel<T>, dim3(static_cast<unsigned>(blocks_rows)), dim3(GR_THREADS), 0, s,
                       total_rows, scale, side, vertices, frame, ptcloud, grid_pt_indexes);
    int st = tpk_launch_status();
    if (st != TPK_OK || total == 0)
        return st;
    hipLaunchKernelGGL(cubic_gather_kernel<T>, dim3(static_cast<unsigned>(blocks)), dim3(GR_THREADS), 0, s, total, n_pts,
                       vertices, channels, cub, cubic_features, grid_pt_indexes, point_features);
    return tpk_launch_status();
}

template <typename T, int LANES>
int launch_spans(int b, int n_pts, int nv, int channels, int64_t cub, const T* grad, const int32_t* indexes, T* grad_maps, hipStream_t s)
{
    int64_t spans = 1;
    while (spans * CubicSpan<T>::CELLS < cub)
        spans *= 2;
    const int64_t blocks = spans * b;
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    const int allowed = tpk_allow_lds(reinterpret_cast<const void*>(cubic_spans_kernel<T, LANES>), sizeof(CubicSpan<T>));
    if (allowed != TPK_OK)
        return allowed;
    hipLaunchKernelGGL((cubic_spans_kernel<T, LANES>), dim3(static_cast<unsigned>(blocks)), dim3(CB_THREADS), sizeof(CubicSpan<T>), s,
                       n_pts, nv, channels, cub, static_cast<int>(spans), grad, indexes, grad_maps);
    return tpk_launch_status();
}

// What the three ways to the gradient of the maps take, in ns beyond a launch (infinite: not possible or not considered).
// Measured over 1 .. 32 clouds of 128 .. 16384 points, 4 .. 128 channels, 4^3 .. 32^3 cells, points spread over the map and over a
// sphere (uneven spans): the way taken is the quicker one or within a tenth of it in 97 of 100 calls.
struct CubicWays
{
    double spans, sums, atomics;
    int64_t group; // channels whose sums a workgroup of cubic_scatter_lds_kernel holds
};

template <typename T>
CubicWays cubic_ways(int b, int channels, int64_t entries, int64_t cub)
{
    CubicWays w{HUGE_VAL, HUGE_VAL, HUGE_VAL, 1};
    const double terms = static_cast<double>(entries) * channels; // of a cloud
    const double bytes = terms * sizeof(T);
    int64_t spans = 1;
    while (spans * CubicSpan<T>::CELLS < cub)
        spans *= 2;
    // Spans: every workgroup looks through all entries of its cloud (0.26 ns each) and adds its own rows (13 ns each), once per
    // CB_CHANNELS channels; offsets into the gradient are 32 bits.
    const bool addressable = bytes < 4294967296.0;
    if (addressable)
    {
        const double rounds = std::max(1.0, static_cast<double>(b) * spans / TPK_COMPUTE_UNITS);
        w.spans = rounds * tpk_ceil_div(channels, CB_CHANNELS) * (5500.0 + entries * (0.26 + 13.0 / spans));
    }
    // Sums in LDS: a workgroup takes a clock or so per sum and three per term; in float64, where the unit keeps up, what counts is
    // whether the gradients of the clouds on a die stay in its 4 MiB of L2.
    const int64_t fit = CS_BYTES / (cub * static_cast<int64_t>(sizeof(T)));
    if (fit > 0)
    {
        // as many channels per workgroup as fit (the fewer workgroups share a line of the gradient, the
        // less often it is read), but a workgroup for every compute unit
        w.group = std::min<int64_t>(fit, channels);
        while (w.group > 1 && b * tpk_ceil_div(channels, w.group) < TPK_COMPUTE_UNITS)
            w.group = (w.group + 1) / 2;
        const double rounds = static_cast<double>(tpk_ceil_div(b * tpk_ceil_div(channels, w.group), TPK_COMPUTE_UNITS));
        const double term = sizeof(T) == 4 ? 1.3 : bytes * tpk_ceil_div(b, 8) > 4194304.0 ? 0.9 : 0.45;
        w.sums = rounds * w.group * (entries * term + cub * 0.13);
    }
    // Atomics in memory, 22 ps of the chip each (25 to 45 where they queue up on few addresses): where a span's
    // look is long and there are many spans.  (32 channels in float32: 8 x 16384 points, 32^3 cells 806 us, sums in LDS 193; 40^3
    // 850, spans 301; 2 x 65536, 32^3 798, sums 766, spans 222; 4 channels, 8 x 16384, 32^3 107, sums 166; 8 channels
    // 240, sums 187.)
    if (!addressable || (spans > 64 && entries > 65536))
        w.atomics = 0.022 * terms * b;
    return w;
}

template <typename T>
int cubic_bwd(int b, int n_pts, int channels, int scale, int neighborhood_size, const T* grad_point_features,
              const int32_t* grid_pt_indexes, T* grad_ptcloud, T* grad_cubic_features, hipStream_t s)
{
    const int64_t nv = cubic_vertices(neighborhood_size);
    if (b < 0 || n_pts < 0 || channels < 0 || scale <= 0 || nv < 0 || scale > 1290)
        return TPK_ERR_INVALID_ARG;
    if (b == 0)
        return TPK_OK;
    const int64_t cub = static_cast<int64_t>(scale) * scale * scale;
    if (channels > 0 && !grad_cubic_features)
        return TPK_ERR_INVALID_ARG;
    // the coordinates only choose the vertices (floor and ceil): their gradient is zero
    // (cuda/src/cubic_feature_sampling_gpu.cu:165-170)
    int st = grad_ptcloud ? fill_zero<T>(static_cast<int64_t>(b) * n_pts * 3, grad_ptcloud, s) : TPK_OK;
    if (st != TPK_OK)
        return st;
    const int64_t entries = static_cast<int64_t>(n_pts) * nv;
    const int64_t total = entries * b * channels;
    if (total > 0 && (!grad_point_features || !grid_pt_indexes))
        return TPK_ERR_INVALID_ARG;
    if (total > 0)
    {
        const CubicWays ways = cubic_ways<T>(b, channels, entries, cub);
        if (ways.spans <= ways.sums && ways.spans <= ways.atomics)
        {
            if (channels > 32)
                return launch_spans<T, 64>(b, n_pts, static_cast<int>(nv), channels, cub, grad_point_features, grid_pt_indexes, grad_cubic_features, s);
            if (channels > 16)
                return launch_spans<T, 32>(b, n_pts, static_cast<int>(nv), channels, cub, grad_point_features, grid_pt_indexes, grad_cubic_features, s);
            return launch_spans<T, 16>(b, n_pts, static_cast<int>(nv), channels, cub, grad_point_features, grid_pt_indexes, grad_cubic_features, s);
        }
        if (ways.sums <= ways.atomics)
        {
            const int64_t blocks = b * tpk_ceil_div(channels, ways.group);
            if (blocks > 0x7fffffffLL)
                return TPK_ERR_UNSUPPORTED;
            const size_t lds = static_cast<size_t>(ways.group * cub) * sizeof(T);
            const int allowed = tpk_allow_lds(reinterpret_cast<const void*>(cubic_scatter_lds_kernel<T>), lds);
            if (allowed != TPK_OK)
                return allowed;
            hipLaunchKernelGGL(cubic_scatter_lds_kernel<T>, dim3(static_cast<unsigned>(blocks)), dim3(CS_THREADS), lds, s, n_pts,
                               static_cast<int>(nv), channels, static_cast<int>(ways.group), cub, grad_point_features, grid_pt_indexes, grad_cubic_features);
            return tpk_launch_status();
        }
    }
    st = fill_zero<T>(static_cast<int64_t>(b) * channels * cub, grad_cubic_features, s);
    if (st != TPK_OK || total == 0)
        return st;
    const int64_t blocks = tpk_ceil_div(total, GR_THREADS);
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(cubic_scatter_kernel<T>, dim3(static_cast<unsigned>(blocks)), dim3(GR_THREADS), 0, s, total, n_pts,
                       static_cast<int>(nv), channels, cub, grad_point_features, grid_pt_indexes, grad_cubic_features);
    return tpk_launch_status();
}

} // namespace

extern "C" int tpk_gridding_f32(int b, int n_pts, float min_x, float max_x, float min_y, float max_y, float min_z,
                                float max_z, const float* ptcloud, float* grid_weights, float* grid_pt_weights,
                                int32_t* grid_pt_indexes, void* stream)
{
    return gridding_native<float>(b, n_pts, min_x, max_x, min_y, max_y, min_z, max_z, ptcloud, grid_weights,
                               grid_pt_weights, grid_pt_indexes, tpk_stream(stream));
}

extern "C" int tpk_gridding_f64(int b, int n_pts, float min_x, float max_x, float min_y, float max_y, float min_z,
                                float max_z, const double* ptcloud, double* grid_weights, double* grid_pt_weights,
                                int32_t* grid_pt_indexes, void* stream)
{
    return gridding_native<double>(b, n_pts, min_x, max_x, min_y, max_y, min_z, max_z, ptcloud, grid_weights,
                                grid_pt_weights, grid_pt_indexes, tpk_stream(stream));
}

extern "C" int tpk_gridding_grad_f32(int b, int n_pts, int n_grid_vertices, const float* grid_pt_weights,
                                     const int32_t* grid_pt_indexes, const float* grad_grid, float* grad_ptcloud,
                                     void* stream)
{
    return gridding_bwd<float>(b, n_pts, n_grid_vertices, grid_pt_weights, grid_pt_indexes, grad_grid, grad_ptcloud,
                               tpk_stream(stream));
}

extern "C" int tpk_gridding_grad_f64(int b, int n_pts, int n_grid_vertices, const double* grid_pt_weights,
                                     const int32_t* grid_pt_indexes, const double* grad_grid, double* grad_ptcloud,
                                     void* stream)
{
    return gridding_bwd<double>(b, n_pts, n_grid_vertices, grid_pt_weights, grid_pt_indexes, grad_grid, grad_ptcloud,
                                tpk_stream(stream));
}

extern "C" int tpk_gridding_batch_f32(int b, int n_pts, double scale, const float* ptcloud, float* grid_weights, void* stream)
{
    return gridding_batch<float>(b, n_pts, scale, ptcloud, grid_weights, nullptr, tpk_stream(stream));
}

extern "C" int tpk_gridding_batch_keep_f32(int b, int n_pts, double scale, const float* ptcloud, float* grid_weights, float* kept, void* stream)
{
    if (b > 0 && n_pts > 0 && !kept)
        return TPK_ERR_INVALID_ARG;
    return gridding_batch<float>(b, n_pts, scale, ptcloud, grid_weights, kept, tpk_stream(stream));
}

extern "C" int tpk_gridding_batch_f64(int b, int n_pts, double scale, const double* ptcloud, double* grid_weights, void* stream)
{
    return gridding_batch<double>(b, n_pts, scale, ptcloud, grid_weights, nullptr, tpk_stream(stream));
}

extern "C" int tpk_gridding_batch_keep_f64(int b, int n_pts, double scale, const double* ptcloud, double* grid_weights, double* kept, void* stream)
{
    if (b > 0 && n_pts > 0 && !kept)
        return TPK_ERR_INVALID_ARG;
    return gridding_batch<double>(b, n_pts, scale, ptcloud, grid_weights, kept, tpk_stream(stream));
}

extern "C" int tpk_gridding_batch_grad_f32(int b, int n_pts, double scale, const float* ptcloud, const float* grad_grid,
                                           float* grad_ptcloud, void* stream)
{
    return gridding_batch_grad<float>(b, n_pts, scale, ptcloud, grad_grid, grad_ptcloud, tpk_stream(stream));
}

extern "C" int tpk_gridding_batch_grad_f64(int b, int n_pts, double scale, const double* ptcloud, const double* grad_grid,
                                           double* grad_ptcloud, void* stream)
{
    return gridding_batch_grad<double>(b, n_pts, scale, ptcloud, grad_grid, grad_ptcloud, tpk_stream(stream));
}

extern "C" size_t tpk_cubic_feature_sampling_workspace_bytes(int b, int n_pts, int channels, int scale, int neighborhood_size,
                                                             int element_bytes)
{
    const int64_t nv = cubic_vertices(neighborhood_size);
    if (b <= 0 || n_pts <= 0 || channels <= 0 || scale <= 0 || scale > 1290 || nv < 0 || (element_bytes != 4 && element_bytes != 8) ||
        !cubic_turns(b, n_pts, channels, scale, nv))
        return 0;
    return static_cast<size_t>(b) * channels * (static_cast<size_t>(scale) * scale * scale) * element_bytes;
}

extern "C" int tpk_cubic_feature_sampling_f32(int b, int n_pts, int channels, int scale, int neighborhood_size,
                                              const float* ptcloud, const float* cubic_features, float* point_features,
                                              int32_t* grid_pt_indexes, void* stream)
{
    return cubic_fwd<float>(b, n_pts, channels, scale, neighborhood_size, false, ptcloud, cubic_features, point_features,
                         grid_pt_indexes, nullptr, 0, tpk_stream(stream));
}

extern "C" int tpk_cubic_feature_sampling_ws_f32(int b, int n_pts, int channels, int scale, int neighborhood_size, int mapped,
                                                const float* ptcloud, const float* cubic_features, float* point_features,
                                                int32_t* grid_pt_indexes, void* workspace, size_t workspace_bytes, void* stream)
{
    return cubic_fwd<float>(b, n_pts, channels, scale, neighborhood_size, mapped != 0, ptcloud, cubic_features, point_features,
                         grid_pt_indexes, workspace, workspace_bytes, tpk_stream(stream));
}

extern "C" int tpk_cubic_feature_sampling_f64(int b, int n_pts, int channels, int scale, int neighborhood_size,
                                              const double* ptcloud, const double* cubic_features, double* point_features,
                                              int32_t* grid_pt_indexes, void* stream)
{
    return cubic_fwd<double>(b, n_pts, channels, scale, neighborhood_size, false, ptcloud, cubic_features, point_features,
                         grid_pt_indexes, nullptr, 0, tpk_stream(stream));
}

extern "C" int tpk_cubic_feature_sampling_ws_f64(int b, int n_pts, int channels, int scale, int neighborhood_size, int mapped,
                                                const double* ptcloud, const double* cubic_features, double* point_features,
                                                int32_t* grid_pt_indexes, void* workspace, size_t workspace_bytes, void* stream)
{
    return cubic_fwd<double>(b, n_pts, channels, scale, neighborhood_size, mapped != 0, ptcloud, cubic_features, point_features,
                         grid_pt_indexes, workspace, workspace_bytes, tpk_stream(stream));
}

extern "C" int tpk_cubic_feature_sampling_grad_f32(int b, int n_pts, int channels, int scale, int neighborhood_size,
                                                   const float* grad_point_features, const int32_t* grid_pt_indexes,
                                                   float* grad_ptcloud, float* grad_cubic_features, void* stream)
{
    return cubic_bwd<float>(b, n_pts, channels, scale, neighborhood_size, grad_point_features, grid_pt_indexes,
                            grad_ptcloud, grad_cubic_features, tpk_stream(stream));
}

extern "C" int tpk_cubic_feature_sampling_grad_f64(int b, int n_pts, int channels, int scale, int neighborhood_size,
                                                   const double* grad_point_features, const int32_t* grid_pt_indexes,
                                                   double* grad_ptcloud, double* grad_cubic_features, void* stream)
{
    return cubic_bwd<double>(b, n_pts, channels, scale, neighborhood_size, grad_point_features, grid_pt_indexes,
                             grad_ptcloud, grad_cubic_features, tpk_stream(stream));
}
