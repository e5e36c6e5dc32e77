// GRNet's two grid operators: gridding (points -> occupancy grid by trilinear weights, and its
// gradient) and cubic feature sampling (features of the grid vertices around a point, and its
// gradient).  Reference: cuda/src/gridding_gpu.cu:29-331, cuda/src/cubic_feature_sampling_gpu.cu:
// 23-210.  The reference runs one block per cloud; here every launch spreads over all points
// (or output elements) of all clouds.  Sums into the grid are float / double atomics in no fixed
// order, as in the reference; the gridding gradient of a point is one thread's sum in the
// reference's order, so it is reproduced bit for bit.
//
// Gridding comes in two forms over the same arithmetic: the reference's native pair, which takes
// coordinates in grid units and hands the factors of every (point, vertex) from the forward to the
// backward pass, and the form of its Python front end (reference gridding.py:34-60) for a whole
// batch at once: coordinates times `factor`, points whose three products sum to zero (padding)
// left out, and a backward pass that forms the factors again from the 12 bytes of a point instead
// of reading the 128 bytes they take.
//
// Vertices outside the grid: the reference forms the linear index regardless (and writes out of
// bounds or into a neighbouring row); here such a vertex gets index -1, adds nothing to the grid
// and contributes no gradient.
#include "tpk_device.h"

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

// cuda/src/gridding_gpu.cu:29-191.  One thread per point, sums in the zeroed grid itself: for grids
// that the kernel below cannot hold, and for more points than its LDS atomics are quick for.
template <typename T>
__global__ __launch_bounds__(GR_THREADS) void gridding_kernel(
    int64_t total_pts, int n_pts, int n_grid_vertices, GridBox box, T factor, bool drop_padding,
    const T* __restrict__ ptcloud, T* __restrict__ grid_weights, T* __restrict__ grid_pt_weights,
    int* __restrict__ grid_pt_indexes)
{
    const int64_t j = static_cast<int64_t>(blockIdx.x) * GR_THREADS + threadIdx.x;
    if (j >= total_pts)
        return;
    T* grid = grid_weights + (j / n_pts) * n_grid_vertices;
    const T px = ptcloud[j * 3 + 0] * factor, py = ptcloud[j * 3 + 1] * factor, pz = ptcloud[j * 3 + 2] * factor;
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
    T* __restrict__ grid_weights, T* __restrict__ grid_pt_weights, int* __restrict__ grid_pt_indexes)
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
        const T px = points[static_cast<int64_t>(i) * 3 + 0] * factor, py = points[static_cast<int64_t>(i) * 3 + 1] * factor;
        const T pz = points[static_cast<int64_t>(i) * 3 + 2] * factor;
        if (drop_padding && is_padding(px, py, pz))
            continue;
        const Trilinear<T> p = trilinear(px, py, pz, box.min_x, box.min_y, box.min_z);
        if (grid_pt_weights && ((i / TPK_WAVE) & (parts - 1)) == part)
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

// cuda/src/cubic_feature_sampling_gpu.cu:23-105.  First kernel: the vertex indices of every
// point (-1 outside the grid); second kernel: one thread per output element, channel fastest.
template <typename T>
__global__ __launch_bounds__(GR_THREADS) void cubic_indexes_kernel(int64_t total_pts, int scale, int neighborhood_size,
                                                                   int n_vertices, const T* __restrict__ ptcloud,
                                                                   int* __restrict__ grid_pt_indexes)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * GR_THREADS + threadIdx.x;
    if (i >= total_pts)
        return;
    int lx, ux, ly, uy, lz, uz;
    planes(ptcloud[i * 3 + 0], &lx, &ux);
    planes(ptcloud[i * 3 + 1], &ly, &uy);
    planes(ptcloud[i * 3 + 2], &lz, &uz);
    const int ns = neighborhood_size - 1;
    int at = 0;
    for (int j = lx - ns; j <= ux + ns; ++j)
        for (int k = ly - ns; k <= uy + ns; ++k)
            for (int m = lz - ns; m <= uz + ns; ++m)
            {
                const bool outside = j < 0 || j >= scale || k < 0 || k >= scale || m < 0 || m >= scale;
                if (at < n_vertices)
                    grid_pt_indexes[i * n_vertices + at] = outside ? -1 : j * scale * scale + k * scale + m;
                ++at;
            }
}

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

// cuda/src/cubic_feature_sampling_gpu.cu:138-175
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

// The same sum with the destination in LDS: a workgroup owns `group` channels of one cloud's
// feature map (group * scale^3 accumulators), walks all (point, vertex) entries of the cloud
// and adds its channels' gradients with LDS atomics, then writes the map out in order.  One
// global atomic per term (a cache line each, at device scope) is what makes the kernel above slow.
constexpr int CS_THREADS = 1024; // LDS atomics are slow: many wavefronts keep the unit busy

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
                 T* grid_pt_weights, int32_t* grid_pt_indexes, hipStream_t s)
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
                           grid_pt_indexes);
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
                       grid_pt_indexes);
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
    return gridding_fwd<T>(b, n_pts, box, T(1), false, ptcloud, grid_weights, grid_pt_weights, grid_pt_indexes, s);
}

// The front end: a grid over [-scale, scale - 1] per axis, coordinates times `scale`.
template <typename T>
int gridding_batch(int b, int n_pts, double scale, const T* ptcloud, T* grid_weights, hipStream_t s)
{
    GridBox box;
    const float lo = static_cast<float>(-scale), hi = static_cast<float>(scale - 1);
    if (b < 0 || n_pts < 0 || !grid_box(lo, hi, lo, hi, lo, hi, &box))
        return TPK_ERR_INVALID_ARG;
    if (b > 0 && (!grid_weights || (n_pts > 0 && !ptcloud)))
        return TPK_ERR_INVALID_ARG;
    return gridding_fwd<T>(b, n_pts, box, static_cast<T>(scale), true, ptcloud, grid_weights, nullptr, nullptr, s);
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

template <typename T>
int cubic_fwd(int b, int n_pts, int channels, int scale, int neighborhood_size, const T* ptcloud,
              const T* cubic_features, T* point_features, int32_t* grid_pt_indexes, hipStream_t s)
{
    const int64_t nv = cubic_vertices(neighborhood_size);
    if (b < 0 || n_pts < 0 || channels < 0 || scale <= 0 || nv < 0 || scale > 1290)
        return TPK_ERR_INVALID_ARG;
    if (b == 0 || n_pts == 0)
        return TPK_OK;
    if (!ptcloud || !grid_pt_indexes || (channels > 0 && (!cubic_features || !point_features)))
        return TPK_ERR_INVALID_ARG;
    const int64_t total_pts = static_cast<int64_t>(b) * n_pts;
    const int64_t total = total_pts * nv * channels;
    const int64_t blocks_pts = tpk_ceil_div(total_pts, GR_THREADS), blocks = tpk_ceil_div(total, GR_THREADS);
    if (blocks > 0x7fffffffLL || nv > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(cubic_indexes_kernel<T>, dim3(static_cast<unsigned>(blocks_pts)), dim3(GR_THREADS), 0, s,
                       total_pts, scale, neighborhood_size, static_cast<int>(nv), ptcloud, grid_pt_indexes);
    int st = tpk_launch_status();
    if (st != TPK_OK || total == 0)
        return st;
    hipLaunchKernelGGL(cubic_gather_kernel<T>, dim3(static_cast<unsigned>(blocks)), dim3(GR_THREADS), 0, s, total, n_pts,
                       static_cast<int>(nv), channels, static_cast<int64_t>(scale) * scale * scale, cubic_features,
                       grid_pt_indexes, point_features);
    return tpk_launch_status();
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
    if ((n_pts > 0 && !grad_ptcloud) || (channels > 0 && !grad_cubic_features))
        return TPK_ERR_INVALID_ARG;
    // the coordinates only choose the vertices (floor and ceil): their gradient is zero
    // (cuda/src/cubic_feature_sampling_gpu.cu:165-170)
    int st = fill_zero<T>(static_cast<int64_t>(b) * n_pts * 3, grad_ptcloud, s);
    if (st != TPK_OK)
        return st;
    const int64_t total = static_cast<int64_t>(b) * n_pts * nv * channels;
    if (total > 0 && (!grad_point_features || !grid_pt_indexes))
        return TPK_ERR_INVALID_ARG;
    // Feature maps that fit in LDS (at least one channel of scale^3 sums in 128 KiB) are summed there.
    const int64_t fit = (128 * 1024) / (cub * static_cast<int64_t>(sizeof(T)));
    if (fit >= 1 && channels > 0 && nv <= 0x7fffffffLL)
    {
        // as many channels per workgroup as fit (the fewer workgroups share a line of the gradient, the
        // less often it is read), but a workgroup for every compute unit
        int64_t group = fit < channels ? fit : channels;
        while (group > 1 && static_cast<int64_t>(b) * tpk_ceil_div(channels, group) < 256)
            group = (group + 1) / 2;
        const int64_t blocks = static_cast<int64_t>(b) * tpk_ceil_div(channels, group);
        if (blocks <= 0x7fffffffLL)
        {
            const size_t lds = static_cast<size_t>(group * cub) * sizeof(T);
            const int allowed = tpk_allow_lds(reinterpret_cast<const void*>(cubic_scatter_lds_kernel<T>), lds);
            if (allowed != TPK_OK)
                return allowed;
            hipLaunchKernelGGL(cubic_scatter_lds_kernel<T>, dim3(static_cast<unsigned>(blocks)), dim3(CS_THREADS), lds, s, n_pts, static_cast<int>(nv), channels,
                               static_cast<int>(group), cub, grad_point_features, grid_pt_indexes, grad_cubic_features);
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
    return gridding_batch<float>(b, n_pts, scale, ptcloud, grid_weights, tpk_stream(stream));
}

extern "C" int tpk_gridding_batch_f64(int b, int n_pts, double scale, const double* ptcloud, double* grid_weights, void* stream)
{
    return gridding_batch<double>(b, n_pts, scale, ptcloud, grid_weights, tpk_stream(stream));
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

extern "C" int tpk_cubic_feature_sampling_f32(int b, int n_pts, int channels, int scale, int neighborhood_size,
                                              const float* ptcloud, const float* cubic_features, float* point_features,
                                              int32_t* grid_pt_indexes, void* stream)
{
    return cubic_fwd<float>(b, n_pts, channels, scale, neighborhood_size, ptcloud, cubic_features, point_features,
                            grid_pt_indexes, tpk_stream(stream));
}

extern "C" int tpk_cubic_feature_sampling_f64(int b, int n_pts, int channels, int scale, int neighborhood_size,
                                              const double* ptcloud, const double* cubic_features,
                                              double* point_features, int32_t* grid_pt_indexes, void* stream)
{
    return cubic_fwd<double>(b, n_pts, channels, scale, neighborhood_size, ptcloud, cubic_features, point_features,
                             grid_pt_indexes, tpk_stream(stream));
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
